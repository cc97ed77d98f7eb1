// Ising checkerboard colour pass on the simple-cubic lattice, multispin
// coded, for any number of chains packed in one arena (a single chain is a
// batch of one).
//
// Replaces the inner loop of MetropolisFlipIntegrator::step and
// MetropolisIntegrator::step (reference src/integrator.rs:66-92, 109-138) with
// the Exchange + Zeeman local energy of src/energy.rs:147-151, 194-206:
// instead of N attempts at uniformly random sites, one sweep updates every
// colour-0 site, then every colour-1 site.
//
// Work item: one 32-position segment of a row, marched through K (the tile, a
// template parameter picked by the host) consecutive z planes, upwards in
// even chunks of K planes and downwards in odd ones.  Along z the row behind
// is the previous row's neighbour ahead, so each plane loads four words (own,
// y-1, y+1, the next plane's) instead of six, and the word that holds the one
// x neighbour outside the segment.  The counts and the decision work on whole
// words (ising_word.hpp).
#include "ising_word.hpp"

#include <type_traits>

namespace vg {

template <uint32_t K, uint32_t MODE>
__global__ __launch_bounds__(256) void ising_sc_pass(const ChainDev* __restrict__ chains,
                                                     const uint32_t* __restrict__ block_chain,
                                                     uint8_t* __restrict__ arena,
                                                     int32_t* __restrict__ partials,
                                                     uint32_t colour, uint32_t s,
                                                     uint32_t total_blocks, uint32_t grid,
                                                     uint32_t opts, uint32_t chain_m) {
    using M = March<6, 1, MODE>;
    constexpr bool PER = M::PER;
    __shared__ uint32_t tie_q[kWaves][kTieRows][M::NREC];
    __shared__ uint32_t thr_q[kWaves][PER ? 1 : 2 * kThrS];
    // opts: bit 0 = falling wave priorities; bits 8-15 = records the tie
    // queue may hold (at most kTieRows; fewer only to exercise the overflow
    // path in tests -- results do not depend on it).
    const uint32_t prio = opts & 1u;
    const uint32_t b = xcd_block(blockIdx.x, grid);
    const ChainDev& C = pass_chain(chains, block_chain, b, total_blocks, opts, chain_m);
    const PassHead h = pass_head(C, b, total_blocks, s);
    const __amdgpu_buffer_rsrc_t ro = plane_rsrc(arena + uniform64(C.off[colour ^ 1u]), h.plane);
    const __amdgpu_buffer_rsrc_t own = plane_rsrc(arena + uniform64(C.off[colour]), h.plane);
    uint32_t (*const q_wave)[M::NREC] = tie_q[threadIdx.x >> 6];
    uint32_t* const thr_wave = thr_q[threadIdx.x >> 6];
    M m(C, h, opts, colour, colour == 1);
    m.load_thresholds(thr_wave);
    if (h.go) {
        const uint32_t ly = h.ly, lz = h.lz, w = h.w, pitch = h.pitch, y = h.y;
        const uint32_t z0 = h.zc * K, nk = min(K, lz - z0);
        const uint32_t i0 = m.i0, nvalid = m.nvalid, vmask = m.vmask;
        const bool px = PER || (h.pbc & 1u), py = PER || (h.pbc & 2u), pz = PER || (h.pbc & 4u);
        const bool ym_ok = y > 0 || py, yp_ok = y + 1 < ly || py;
        // offsets of rows y-1 and y+1 relative to row y (wrapping when periodic)
        const uint32_t dym = y > 0 ? 0u - pitch : (ly - 1) * pitch;
        const uint32_t dyp = y + 1 < ly ? pitch : 0u - (ly - 1) * pitch;
        const uint32_t gy = (ym_ok ? 0u : 1u) + (yp_ok ? 0u : 1u);
        // x neighbours of position i: i-1, i (q = 0) or i, i+1 (q = 1) in the
        // other plane's same row; q alternates from plane to plane.  The one
        // outside the segment is position i0-1, or w-1 across the periodic end
        // (q = 0), or i0+32, or position 0 (q = 1), which lands in the bit of
        // the last valid position; it reads 0 when x is open there, and then
        // xe is its site, the one with an absent x slot (32: none).
        const bool xr_in = i0 + kIsingSeg < w;
        const XPos x0 = xpos(i0 > 0 ? i0 - 1 : w - 1);
        const XPos x1 = xpos(xr_in ? i0 + kIsingSeg : 0u);
        const bool xok0 = i0 > 0 || px, xok1 = xr_in || px;
        const uint32_t xe0 = xok0 ? 32u : 0u, xe1 = xok1 ? 32u : nvalid - 1u;
        const uint32_t xr_sh = xr_in ? 31u : nvalid - 1u;
        // Even z chunks march up, odd ones down: two chunks meeting at a seam
        // then read the seam planes in the same step, and the L2 fetches
        // those rows once.
        const bool down = h.zc & 1u;
        const uint32_t zstep = ly * pitch;  // bytes between planes z and z+1
        const uint32_t step = down ? 0u - zstep : zstep;
        // Along the march: the plane ahead of plane z is z + 1 (up) or z - 1
        // (down), or across the periodic end from the lattice's last (up) or
        // first (down) plane, where it is absent when z is open.
        const uint32_t zend = down ? 0u : lz - 1u;
        const uint32_t wrap = down ? (lz - 1) * zstep : 0u - (lz - 1) * zstep;
        uint32_t z = down ? z0 + nk - 1u : z0;
        uint32_t row = y + ly * z;
        uint32_t rowoff = row * pitch;  // this row
        const uint32_t woff = i0 >> 3;
        // the row window along z: the plane behind the march and the current
        // one (from the march's first plane, behind is the far end's plane)
        const uint32_t zbeg = down ? lz - 1u : 0u;
        bool behind_ok = z != zbeg || pz;
        const uint32_t back = z != zbeg ? rowoff + woff - step : rowoff + woff - wrap;
        uint32_t behind = load_word(ro, behind_ok ? back : kNoRow);
        uint32_t here = load_word(ro, rowoff + woff);
        uint32_t qm = 0u - ((colour + y + z) & 1u);  // q as a mask
        const uint32_t wA = ctr_w(h.t, kIsingA, colour);
        // A plane's words as loaded; loads of the march's next plane are in
        // flight while a plane is decided.
        struct Plane {
            uint32_t own, ym, yp, ab;
            uint32_t x;
        };
        const auto load_plane = [&](uint32_t pz_, uint32_t roff, uint32_t q, bool in) {
            const uint32_t off = roff + woff;
            const bool at_end = pz_ == zend;
            const bool ahead_ok = !at_end || pz;
            const uint32_t ahead_off = at_end ? off + wrap : off + step;
            const bool xok = q ? xok1 : xok0;
            Plane p;
            p.own = load_word(own, in ? off : kNoRow);
            p.ym = load_word(ro, in && ym_ok ? off + dym : kNoRow);
            p.yp = load_word(ro, in && yp_ok ? off + dyp : kNoRow);
            p.ab = load_word(ro, in && ahead_ok ? ahead_off : kNoRow);
            p.x = load_word(ro, in && xok ? roff + (q ? x1.off : x0.off) : kNoRow);
            return p;
        };
        Plane next = load_plane(z, rowoff, qm, true);
        const auto plane = [&](auto plain, uint32_t k) {
            constexpr bool PLAIN = decltype(plain)::value;
            // The SIMD arbiter favours older waves; when every wave of the
            // pass is resident at once, a wave's priority falls as it
            // marches, so the waves of a SIMD progress together and the pass
            // does not end in a tail of a few young waves.
            if (prio) set_prio(((K - 1u - k) * 4u) / K);
            const Plane cur = next;
            const uint32_t off = rowoff + woff;
            const bool ahead_ok = z != zend || pz;
            const uint32_t znext = down ? z - 1u : z + 1u;
            if (k + 1 < K) next = load_plane(znext, rowoff + step, ~qm, k + 1 < nk);

            Edge ed{0u, 1u, 32u, 0u, 0u};
            if constexpr (!PER) {
                ed.g = gy + (behind_ok ? 0u : 1u) + (ahead_ok ? 0u : 1u);
                ed.xe = qm ? xe1 : xe0;
            }
            const uint32_t gw = m.template wave_absent<PLAIN>(ed);

            // draws first: they do not wait for the loads
            const U4 r0 = philox(U4{i0 >> 4, row, (uint32_t)h.t, wA}, h.k0, h.k1);
            const U4 r1 = philox(U4{(i0 >> 4) + 1u, row, (uint32_t)h.t, wA}, h.k0, h.k1);
            uint32_t d[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
            keep_draws(d);

            const uint32_t o = arrived(cur.own);
            uint32_t nym = arrived(cur.ym), nyp = arrived(cur.yp);
            const uint32_t ahead = arrived(cur.ab);
            const uint32_t xbit = (arrived(cur.x) >> (qm ? x1.sh : x0.sh)) & 1u;
            const uint32_t no = ~o;
            const uint32_t xa = here & vmask;
            uint32_t xb = bop3<kSel>((xa >> 1) | (xbit << xr_sh), (xa << 1) | xbit, qm);
            uint32_t nzm = behind, nzp = ahead;
            if constexpr (!PER) {
                // an absent neighbour counts as anti-aligned with its site
                const uint32_t eb = ed.xe < 32u ? 1u << ed.xe : 0u;
                xb = bop3<kSel>(no, xb, eb);
                nym = ym_ok ? nym : no;
                nyp = yp_ok ? nyp : no;
                nzm = behind_ok ? nzm : no;
                nzp = ahead_ok ? nzp : no;
            }
            // aligned count a = 0..6: neighbour n is aligned where n ^ no is
            // set.  Two full adders over triples of neighbours (a full
            // adder's outputs for complemented inputs are the complements, so
            // the alignment goes in after them), then their sum.
            const uint32_t s1 = bop3<kXor3>(xa, xb, nym), c1 = bop3<kMaj3>(xa, xb, nym);
            const uint32_t s2 = bop3<kXor3>(nyp, nzm, nzp), c2 = bop3<kMaj3>(nyp, nzm, nzp);
            const uint32_t hc = bop3<0x42>(s1, s2, no);  // (s1 ^ no) & (s2 ^ no)
            uint32_t a[3];
            a[0] = s1 ^ s2;
            a[1] = bop3<kXor3>(c1, c2, hc);
            a[2] = bop3<kSel>(hc, c1 ^ no, c1 ^ c2);  // maj(c1 ^ no, c2 ^ no, hc)
            m.template word<PLAIN>(own, q_wave, thr_wave, gw, o, a, nullptr, d, ed, off, row);
            behind = here;
            here = ahead;
            behind_ok = true;
            rowoff += step;
            z = znext;
            row = down ? row - ly : row + ly;
            qm = ~qm;
        };
        // The plain plan's march is unrolled (no loop code, no register copies
        // for the loads in flight).
        if (h.plain) {
            m.load_masks();
#pragma unroll
            for (uint32_t k = 0; k < K; ++k) {
                if (k >= nk) break;
                plane(std::true_type{}, k);
            }
        } else {
#pragma unroll 1
            for (uint32_t k = 0; k < nk; ++k) plane(std::false_type{}, k);
        }
        m.fold(nk, 0u);
    }
    m.settle_queue(own, q_wave, h.pitch, 0u);
    m.partials(partials, (uint64_t)(s * 2u + colour) * total_blocks + b, h.active);
}

#define VG_SC_PASS(K, MODE)                                                                     \
    template __global__ void ising_sc_pass<K, MODE>(const ChainDev*, const uint32_t*, uint8_t*, \
                                                    int32_t*, uint32_t, uint32_t, uint32_t,     \
                                                    uint32_t, uint32_t, uint32_t);
VG_SC_PASS(1, kOpen)
VG_SC_PASS(2, kOpen)
VG_SC_PASS(4, kOpen)
VG_SC_PASS(8, kOpen)
VG_SC_PASS(1, kPeriodic)
VG_SC_PASS(2, kPeriodic)
VG_SC_PASS(4, kPeriodic)
VG_SC_PASS(8, kPeriodic)
#undef VG_SC_PASS

// grid = (chains, sweeps).
__global__ __launch_bounds__(1024) void ising_reduce(const ChainDev* __restrict__ chains,
                                                    const int32_t* __restrict__ partials,
                                                    uint32_t total_blocks, uint32_t ncol,
                                                    uint32_t nsw, int64_t* __restrict__ records) {
    reduce_sweep(chains[blockIdx.x], partials, total_blocks, ncol, nsw, blockIdx.y, records);
}

}  // namespace vg
