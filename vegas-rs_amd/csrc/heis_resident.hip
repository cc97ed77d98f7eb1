// Whole sweep blocks of small Heisenberg chains, one workgroup a chain, spins
// in LDS.
//
// The same sweeps as the colour passes (heis_sc.hip and its bcc and fcc
// siblings), the same draws, the same fp32 operations in the same order, the
// same sums.  A pass of a small chain is one wave a SIMD at most and lasts as
// long as that wave issues its 1100 instructions, one every 8 cycles: 6.6 us
// whatever the size.  Three quarters of them make the proposals, which depend
// on the site and the sweep and not on the spins.  So a sweep block is two
// launches:
//   heis_draws fills a workspace with the proposal and the acceptance uniform
//     of every site of many sweeps, one lane each, on the whole chip (flip
//     proposals: the uniform alone);
//   heis_resident runs those sweeps, one workgroup a chain, a lane a site (R
//     sites past 1024 a colour): spins as {x, y, z, -} in LDS, neighbours at
//     indices worked out once, the next colour's draws in flight meanwhile.
//
// us a sweep of one chain with random proposals, by passes and here: sc 8^3
// 11.6, 2.2; 16^3 13.0, 4.3; 20^3 13.1, 7.0; bcc 8^3 13.0, 2.6; fcc 8^3 26.1,
// 4.2; 12^3 27.0, 9.0.  A sweep is then a workgroup's: its one CU issues the
// update's instructions, about 90 a site, and below 12^3 waits for LDS and the
// barrier.
#include "heis_common.hpp"
#include "resident.hpp"

namespace vg {

// Draws of the sweeps s0 .. s0 + ns - 1 of the block: entry ((k * ns + s) *
// ncol + c) * nc + site of chain k, chains `stride` entries of ns sweeps apart.
// grid (sites of a colour, ns * ncol, chains).
__global__ __launch_bounds__(256) void heis_draws(const ChainDev* __restrict__ chains, uint32_t s0,
                                                  uint32_t ns, uint32_t stride,
                                                  float4* __restrict__ out) {
    const ChainDev& C = chains[blockIdx.z];
    const uint32_t w = C.w, nc = C.rows * w, ncol = C.ncol;
    const uint32_t site = blockIdx.x * 256u + threadIdx.x;
    const uint32_t s = blockIdx.y / ncol, c = blockIdx.y - s * ncol;
    if (site >= nc || s >= ns || s0 + s >= C.limit) return;
    const uint32_t row = site / w, i = site - row * w;
    const uint64_t t = C.sweep0 + s0 + s;
    float u, p[3] = {0.0f, 0.0f, 0.0f};
    const uint64_t at = (uint64_t)blockIdx.z * stride * ns + (uint64_t)blockIdx.y * nc + site;
    if (C.proposal) {
        if (!proposal_first(C.seed, i, row, t, c, u, p)) proposal_rest(C.seed, i, row, t, c, p);
        out[at] = make_float4(p[0], p[1], p[2], u);
    } else {
        u = unit24(u4_word(flip_words(C.seed, i, row, t, c), i & 3u));
        out[at].w = u;
    }
}

// WIDE: a lane adds up to eight sites' terms a sweep in int32 multiples of 2^-27,
// exact while each is below 2, as they are with spins and an anisotropy axis of
// length 1.  For longer ones the sums are 64-bit (the passes' items hold four
// sites).  (So for every chain: sc 20^3 5% and fcc 12^3 7% more a sweep; a branch
// in one kernel, 3 to 8%.)
template <uint32_t Z, uint32_t R, bool WIDE>
__global__ __launch_bounds__(kResidentBlock) void heis_resident(
    const ChainDev* __restrict__ chains, float* __restrict__ arena, uint32_t s0, uint32_t ns,
    uint32_t stride, const float4* __restrict__ draws, uint32_t nsw,
    int64_t* __restrict__ records) {
    constexpr uint32_t NCOL = Z == 12 ? 4 : 2;
    extern __shared__ __align__(16) uint8_t lds[];
    const ChainDev& C = chains[blockIdx.x];
    if (s0 >= C.limit) return;
    const uint32_t run = min(ns, C.limit - s0);
    const uint32_t tid = threadIdx.x, block = blockDim.x;
    const uint32_t w = C.w, nc = C.rows * w, n = NCOL * nc;
    const bool rnd = C.proposal != 0;
    float4* const spin = reinterpret_cast<float4*>(lds);
    int64_t* const sums = reinterpret_cast<int64_t*>(spin + n + 1u);
    const float4* const mine = draws + (uint64_t)blockIdx.x * stride * ns;

    const uint64_t plane = C.plane;
    for (uint32_t k = tid; k < n; k += block) {
        const uint32_t c = k / nc, site = k - c * nc, row = site / w;
        const float* const at = arena + C.off[c] + (uint64_t)row * C.pitch + (site - row * w);
        spin[k] = make_float4(at[0], at[plane], at[2 * plane], 0.0f);
    }
    if (tid == 0) spin[n] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // the absent neighbour
    for (uint32_t k = tid; k < 5u * run; k += block) sums[k] = 0;

    uint32_t nbr[NCOL][R][Z / 2];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        const uint32_t site = min(tid + r * block, nc - 1u);
        const uint32_t row = site / w, i = site - row * w;
        const uint32_t z = fast_div(row, C.ly_m, C.ly_s), y = row - z * C.ly;
#pragma unroll
        for (uint32_t c = 0; c < NCOL; ++c)
#pragma unroll
            for (uint32_t d = 0; d < Z / 2; ++d)
                nbr[c][r][d] = neighbour_at<Z>(C, c, y, z, i, 2u * d, nc, n) |
                               neighbour_at<Z>(C, c, y, z, i, 2u * d + 1u, nc, n) << 16;
    }
    // the draws of the next colour, in flight while a colour is updated
    float4 next[R];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
        next[r] = mine[min(tid + r * block, nc - 1u)];
    __syncthreads();

    for (uint32_t s = 0; s < run; ++s) {
        int32_t s32[4] = {0, 0, 0, 0};
        int64_t s64[4] = {0, 0, 0, 0}, bsum = 0;
#pragma unroll
        for (uint32_t c = 0; c < NCOL; ++c) {
            float4 d[R];
            const uint32_t half = min(s * NCOL + c + 1u, run * NCOL - 1u);
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                d[r] = next[r];
                next[r] = mine[half * nc + min(tid + r * block, nc - 1u)];
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t site = tid + r * block;
                if (site >= nc) break;
                const float4 own = spin[c * nc + site];
                const float o[3] = {own.x, own.y, own.z};
                float h[3], hb[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
                for (uint32_t k = 0; k < Z; ++k) {
                    const uint32_t both = nbr[c][r][k / 2];
                    const float4 v = spin[k & 1u ? both >> 16 : both & 0xFFFFu];
                    h[0] = k ? fa(h[0], v.x) : v.x;
                    h[1] = k ? fa(h[1], v.y) : v.y;
                    h[2] = k ? fa(h[2], v.z) : v.z;
                    if (Z == 12 && k + 1u == 4u * c) {
                        hb[0] = h[0];
                        hb[1] = h[1];
                        hb[2] = h[2];
                    }
                }
                const float p[3] = {rnd ? d[r].x : -o[0], rnd ? d[r].y : -o[1],
                                    rnd ? d[r].z : -o[2]};
                float m[3];
                heis_update(C, c > 0, o, h, Z == 12 ? hb : h, d[r].w, p, m, s32, bsum);
                spin[c * nc + site] = make_float4(m[0], m[1], m[2], 0.0f);
                if (WIDE)
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) {
                        s64[k] += s32[k];
                        s32[k] = 0;
                    }
            }
            __syncthreads();
        }
        // At most R * NCOL sites a lane, each below 2^31: within wave_sum_split's
        // bounds.
        int64_t v[5];
        v[0] = wave_sum_split(bsum);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) v[1 + k] = wave_sum_split(WIDE ? s64[k] : s32[k]);
        if ((tid & 63u) == 0u)
#pragma unroll
            for (uint32_t k = 0; k < 5; ++k)
                atomicAdd(reinterpret_cast<unsigned long long*>(sums + 5u * s + k),
                          (unsigned long long)v[k]);
    }
    __syncthreads();
    for (uint32_t k = tid; k < 5u * run; k += block)
        records[((uint64_t)C.slot * nsw + s0) * 5u + k] = sums[k];
    for (uint32_t k = tid; k < n; k += block) {
        const uint32_t c = k / nc, site = k - c * nc, row = site / w;
        float* const at = arena + C.off[c] + (uint64_t)row * C.pitch + (site - row * w);
        const float4 v = spin[k];
        at[0] = v.x;
        at[plane] = v.y;
        at[2 * plane] = v.z;
    }
}

#define VG_HEIS_RESIDENT_OF(Z, R, WIDE)                                                          \
    template __global__ void heis_resident<Z, R, WIDE>(const ChainDev*, float*, uint32_t,        \
                                                       uint32_t, uint32_t, const float4*,        \
                                                       uint32_t, int64_t*);
#define VG_HEIS_RESIDENT(Z, R)        \
    VG_HEIS_RESIDENT_OF(Z, R, false)  \
    VG_HEIS_RESIDENT_OF(Z, R, true)
VG_HEIS_RESIDENT(6, 1)
VG_HEIS_RESIDENT(6, 2)
VG_HEIS_RESIDENT(6, 4)
VG_HEIS_RESIDENT(8, 1)
VG_HEIS_RESIDENT(8, 2)
VG_HEIS_RESIDENT(8, 4)
VG_HEIS_RESIDENT(12, 1)
VG_HEIS_RESIDENT(12, 2)
#undef VG_HEIS_RESIDENT
#undef VG_HEIS_RESIDENT_OF

}  // namespace vg
