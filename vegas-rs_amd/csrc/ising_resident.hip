// Whole sweep blocks of small Ising chains, one workgroup a chain, spins in
// LDS.
//
// The same sweeps as the colour passes (MetropolisFlipIntegrator::step /
// MetropolisIntegrator::step, reference src/integrator.rs:66-138, with the
// Exchange + Zeeman local energy of src/energy.rs:147-151, 194-206), the same
// draws and the same sums.  A pass of a small chain lasts about 3 us whatever
// its size: the launch, a cold descriptor, and a few waves that issue one
// instruction every 8 cycles through a pass's start-up.  Here a chain's sweeps
// are a loop of one workgroup, with nothing to launch and nothing to read back
// between them:
//   - the draws depend on the site and the sweep only, not on the spins, so
//     the workgroup makes those of as many sweeps as its LDS holds at once,
//     all its lanes busy whatever the chain's size, each site's 32 bits whole
//     (no ties to settle);
//   - a colour update is then one lane a site: the class sum S from the
//     neighbours' bytes, at addresses worked out once (two 16-bit ones a
//     register), a threshold from a table, the new byte.  About 30
//     instructions and two LDS round trips, and a barrier (a wave's own LDS
//     order where a colour fits one wave).
// A spin is a byte 0 (Down) or 16 (Up) and an absent neighbour a byte 8: the sum
// of the neighbours' bytes is 8 S, the byte offset of class S in a table row, and
// the sum of the present neighbours' spins is S - Z.
//
// us a sweep of one chain, by passes and here: sc 10 x 10 x 2 5.8, 0.7; 8^3
// 6.0, 0.9; 16^3 7.0, 2.3; 20^3 7.3, 4.7; bcc 4^3 6.2, 0.5; 8^3 7.0, 1.0; 16^3
// 7.8, 4.6; fcc 8^3 14.9, 1.6; 12^3 16.1, 3.7.  At 8^3 the two LDS round trips
// and the barrier of each colour are most of it; from about 12^3 the
// instructions, of the draws two thirds.
#include "resident.hpp"

namespace vg {

namespace {

// Entries of a table row: the rows of the two bits are 16 * kUp bytes apart, kUp
// an Up spin's byte.
constexpr uint32_t kUp = 16, kRow = 2 * kUp;

// LDS of a chain, in bytes: its spins with the absent neighbour's byte, the
// threshold table, then per sweep its sums, draws and proposals.
__host__ __device__ constexpr uint32_t resident_spins(uint32_t n) { return (n + 16u) & ~15u; }

}  // namespace

// R: sites of a colour per lane.  With one, sc and bcc keep within the
// registers of two workgroups a CU (512 chains of sc 8^3: 2.31 us a sweep, now
// 1.76); fcc spills there (8^3 2.0 us a sweep, 2.2).  lds_bytes: the launch's dynamic LDS.
// SOLO: the colours of the group's chains have at most 64 sites and one wave
// updates them: its LDS operations are in order, so it needs no barrier, and it
// leaves its lanes' sums for the other waves to reduce with it when a batch is
// done (10 x 10, 1000 sweeps: 622 us in the general form, 406 so).
template <uint32_t Z, uint32_t R, bool SOLO>
__global__ __launch_bounds__(kResidentBlock, Z < 12 && R == 1 ? 8 : 4) void ising_resident(
    const ChainDev* __restrict__ chains, uint8_t* __restrict__ arena, uint32_t nsw,
    uint32_t lds_bytes, int64_t* __restrict__ records) {
    constexpr uint32_t NCOL = Z == 12 ? 4 : 2;
    extern __shared__ __align__(16) uint8_t lds[];
    const ChainDev& C = chains[blockIdx.x];
    const uint32_t tid = threadIdx.x;
    const uint32_t run = min(nsw, C.limit);
    if (!run) return;
    const uint32_t w = C.w, segs = C.segs, nc = C.rows * w, n = NCOL * nc;
    const uint32_t words = C.rows * segs;  // of a colour
    const bool rnd = C.proposal != 0;
    const uint32_t k0 = (uint32_t)C.seed, k1 = (uint32_t)(C.seed >> 32);
    uint8_t* const spin = lds;
    uint2* const table = reinterpret_cast<uint2*>(lds + resident_spins(n));
    int32_t* const sums = reinterpret_cast<int32_t*>(table + 2u * kRow);
    // sweeps whose draws are held at once
    const uint32_t per_sweep = (SOLO ? 256u : 8u) + n * (rnd ? 5u : 4u);
    const uint32_t room = lds_bytes - resident_spins(n) - 2u * kRow * 8u;
    const uint32_t batch = min(run, room / per_sweep);
    uint32_t* const draw = reinterpret_cast<uint32_t*>(sums + (SOLO ? 64u : 2u) * batch);
    uint8_t* const prop = reinterpret_cast<uint8_t*>(draw + n * batch);

    // Spins, the absent neighbour, the table {threshold, always accepted}.
    for (uint32_t k = tid; k < NCOL * words; k += kResidentBlock) {
        const uint32_t c = k / words, at = k - c * words;
        const uint32_t row = fast_div(at, C.segs_m, C.segs_s), i0 = (at - row * segs) * kIsingSeg;
        uint32_t v = *reinterpret_cast<const uint32_t*>(arena + C.off[c] +
                                                        (uint64_t)row * C.pitch + (i0 >> 3));
        uint8_t* const out = spin + c * nc + row * w + i0;
        const uint32_t m = min(kIsingSeg, w - i0);
        for (uint32_t j = 0; j < m; ++j) out[j] = (uint8_t)(((v >> j) & 1u) << 4);
    }
    if (tid == 0) spin[n] = 8;
    for (uint32_t k = tid; k < 2u * kThrS; k += kResidentBlock) {
        const uint32_t b = k / kThrS, S = k - b * kThrS;
        table[b * kRow + S] = make_uint2(C.thr[b][S], (C.always[b] >> S) & 1u);
    }

    // The lane's sites and their neighbours' addresses.
    // With one site a lane there are registers for an address each.
    constexpr bool kWide = R == 1;
    uint32_t nbr[NCOL][R][kWide ? Z : Z / 2];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        const uint32_t site = min(tid + r * kResidentBlock, nc - 1u);
        const uint32_t row = site / w, i = site - row * w;
        const uint32_t z = fast_div(row, C.ly_m, C.ly_s), y = row - z * C.ly;
#pragma unroll
        for (uint32_t c = 0; c < NCOL; ++c)
#pragma unroll
            for (uint32_t d = 0; d < Z; ++d) {
                const uint32_t at = neighbour_at<Z>(C, c, y, z, i, d, nc, n);
                if (kWide)
                    nbr[c][r][d] = at;
                else
                    nbr[c][r][d / 2] = d & 1u ? nbr[c][r][d / 2] | at << 16 : at;
            }
    }

    const uint32_t dw = kResidentBlock % words, dh = kResidentBlock / words;
    for (uint32_t done = 0; done < run; done += batch) {
        const uint32_t ns = min(batch, run - done);
        const uint64_t t0 = C.sweep0 + done;
        // The draws of ns sweeps, a lane a word of positions.
        uint32_t half = tid / words, at = tid - half * words;
        while (half < ns * NCOL) {
            const uint32_t s = half / NCOL, c = half % NCOL;
            const uint64_t t = t0 + s;
            const uint32_t row = fast_div(at, C.segs_m, C.segs_s);
            const uint32_t i0 = (at - row * segs) * kIsingSeg, m = min(kIsingSeg, w - i0);
            const uint32_t wA = ctr_w(t, kIsingA, c), wB = ctr_w(t, kIsingB, c);
            const U4 r0 = philox(U4{i0 >> 4, row, (uint32_t)t, wA}, k0, k1);
            const U4 r1 = Z == 6 || m > 16u
                              ? philox(U4{(i0 >> 4) + 1u, row, (uint32_t)t, wA}, k0, k1)
                              : r0;
            uint32_t* const dr = draw + half * nc + row * w + i0;
#pragma unroll
            for (uint32_t j0 = 0; j0 < kIsingSeg; j0 += 4u) {
                if (j0 >= m) break;
                const U4 rb = philox(U4{(i0 + j0) >> 2, row, (uint32_t)t, wB}, k0, k1);
                // the high bytes of sites j0 .. j0+3, a byte each
                uint32_t hi = 0;
                if constexpr (Z == 6) {
                    // bit j of the calls' word k is bit k of site j's byte
                    const uint32_t p[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
                    for (uint32_t k = 0; k < 8; ++k) {
                        const uint32_t nib = (p[k] >> j0) & 15u;
                        hi |= ((nib * 0x00204081u) & 0x01010101u) << k;
                    }
                } else {
                    hi = u4_word(j0 < 16u ? r0 : r1, (j0 & 15u) >> 2);
                }
                const uint32_t q[4] = {rb.x, rb.y, rb.z, rb.w};
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e)
                    if (j0 + e < m) dr[j0 + e] = (((hi >> (8u * e)) & 255u) << 24) | (q[e] >> 8);
            }
            if (rnd) {
                const U4 rp = philox(U4{i0 >> 7, row, (uint32_t)t, ctr_w(t, kIsingProposal, c)}, k0,
                                     k1);
                const uint32_t v = u4_word(rp, (i0 >> 5) & 3u);
                uint8_t* const pr = prop + half * nc + row * w + i0;
                for (uint32_t j = 0; j < m; ++j) pr[j] = (uint8_t)((~(v >> j) & 1u) << 4);
            }
            half += dh;
            at += dw;
            if (at >= words) {
                at -= words;
                ++half;
            }
        }
        if (!SOLO)
            for (uint32_t k = tid; k < 2u * ns; k += kResidentBlock) sums[k] = 0;
        __syncthreads();

        if (!SOLO || tid < 64u) {
            for (uint32_t s = 0; s < ns; ++s) {
                int32_t acc = 0;  // bond sum << 16 + magnetisation (both small)
#pragma unroll
                for (uint32_t c = 0; c < NCOL; ++c) {
                    const uint32_t base = (s * NCOL + c) * nc;
#pragma unroll
                    for (uint32_t r = 0; r < R; ++r) {
                        const uint32_t site = tid + r * kResidentBlock;
                        if (site >= nc) break;
                        const uint32_t d = draw[base + site];
                        const uint32_t own = spin[c * nc + site];
                        uint32_t S8 = 0, low = 0;
#pragma unroll
                        for (uint32_t k = 0; k < Z; ++k) {
                            const uint32_t at = kWide ? nbr[c][r][k]
                                                      : (k & 1u ? nbr[c][r][k / 2] >> 16
                                                                : nbr[c][r][k / 2] & 0xFFFFu);
                            S8 += spin[at];
                            if (Z == 12 && k + 1u == 4u * c) low = S8;
                        }
                        const uint2 e = *reinterpret_cast<const uint2*>(
                            reinterpret_cast<const uint8_t*>(table) + (own * kUp + S8));
                        bool ok = (d < e.x) | (e.y != 0u);
                        if (rnd) ok = ok & (prop[base + site] != own);
                        const uint32_t now = ok ? own ^ kUp : own;
                        spin[c * nc + site] = (uint8_t)now;
                        const int32_t v = (int32_t)(now >> 3) - 1;
                        acc += v;
                        // the bonds to lower colours
                        if (Z == 12 ? c > 0 : c == 1)
                            acc += v * ((int32_t)((Z == 12 ? low : S8) << 13) -
                                        (int32_t)(Z == 12 ? 4u * c : Z) * 65536);
                    }
                    if (SOLO) {
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    } else {
                        __syncthreads();
                    }
                }
                if (SOLO) {
                    sums[64u * s + tid] = acc;
                    continue;
                }
                acc = wave_total(acc);
                if ((tid & 63u) == 63u && tid - 63u < nc) {
                    const int32_t m = (int16_t)acc;
                    atomicAdd(&sums[2u * s], m);
                    atomicAdd(&sums[2u * s + 1u], (acc - m) >> 16);
                }
            }
        }
        __syncthreads();
        const auto record = [&](uint32_t s, int32_t m, int32_t bond) {
            int64_t* const rec = records + ((uint64_t)C.slot * nsw + done + s) * 5u;
            rec[0] = bond;
            rec[1] = 0;
            rec[2] = 0;
            rec[3] = m;
            rec[4] = 0;
        };
        if (SOLO) {
            for (uint32_t s = tid >> 6; s < ns; s += kResidentBlock / 64u) {
                const int32_t acc = wave_total(sums[64u * s + (tid & 63u)]);
                const int32_t m = (int16_t)acc;
                if ((tid & 63u) == 63u) record(s, m, (acc - m) >> 16);
            }
        } else {
            for (uint32_t s = tid; s < ns; s += kResidentBlock)
                record(s, sums[2u * s], sums[2u * s + 1u]);
        }
        __syncthreads();
    }

    for (uint32_t k = tid; k < NCOL * words; k += kResidentBlock) {
        const uint32_t c = k / words, at = k - c * words;
        const uint32_t row = fast_div(at, C.segs_m, C.segs_s), i0 = (at - row * segs) * kIsingSeg;
        const uint8_t* const in = spin + c * nc + row * w + i0;
        const uint32_t m = min(kIsingSeg, w - i0);
        uint32_t v = 0;
        for (uint32_t j = 0; j < m; ++j) v |= ((uint32_t)in[j] >> 4) << j;
        *reinterpret_cast<uint32_t*>(arena + C.off[c] + (uint64_t)row * C.pitch + (i0 >> 3)) = v;
    }
}

#define VG_RESIDENT(Z, R, SOLO)                                                                 \
    template __global__ void ising_resident<Z, R, SOLO>(const ChainDev*, uint8_t*, uint32_t,    \
                                                        uint32_t, int64_t*);
VG_RESIDENT(6, 1, true)
VG_RESIDENT(6, 1, false)
VG_RESIDENT(6, 2, false)
VG_RESIDENT(6, 4, false)
VG_RESIDENT(8, 1, true)
VG_RESIDENT(8, 1, false)
VG_RESIDENT(8, 2, false)
VG_RESIDENT(8, 4, false)
VG_RESIDENT(12, 1, true)
VG_RESIDENT(12, 1, false)
VG_RESIDENT(12, 2, false)
#undef VG_RESIDENT

}  // namespace vg
