// Ising checkerboard colour pass on the body-centred cubic lattice, multispin
// coded, for any number of chains packed in one arena.
//
// The same update as the simple-cubic pass (MetropolisFlipIntegrator::step /
// MetropolisIntegrator::step, reference src/integrator.rs:66-138, with the
// Exchange + Zeeman local energy of src/energy.rs:147-151, 194-206) on the
// bcc topology: the two colours are the two sublattices.  A corner site of
// cell (x,y,z) (colour 0) bonds to the body centres of cells (x-dx, y-dy,
// z-dz), a body centre (colour 1) to the corners of cells (x+dx, y+dy, z+dz),
// dx,dy,dz in {0,1}: four rows of the other plane, each at positions x and
// x-1 (colour 0) or x and x+1 (colour 1).
//
// Work item: one 32-position segment of a row, marched up through K (the
// tile) consecutive z planes.  The four neighbour rows of plane z are two
// pairs, (y, zl), (y', zl) and (y, zu), (y', zu), with (zl, zu) = (z-1, z) for
// colour 0 and (z, z+1) for colour 1; the upper pair of plane z is the lower
// pair of plane z+1, so a plane loads its own word and one pair (two words
// and the two that hold their x neighbour outside the segment) and adds the
// pair's counts (0..4, three planes, from one full and one half adder) to
// those kept from the plane before.  Counts and decision work on whole words
// (ising_word.hpp).
#include "ising_word.hpp"

#include <type_traits>

namespace vg {

template <uint32_t A, uint32_t K, uint32_t MODE>
__global__ __launch_bounds__(256) void ising_bcc_pass(const ChainDev* __restrict__ chains,
                                                      const uint32_t* __restrict__ block_chain,
                                                      uint8_t* __restrict__ arena,
                                                      int32_t* __restrict__ partials, uint32_t s,
                                                      uint32_t total_blocks, uint32_t grid,
                                                      uint32_t opts, uint32_t chain_m) {
    using M = March<8, A == 1 ? 1 : 0, MODE>;
    constexpr bool PER = M::PER;
    __shared__ uint32_t tie_q[kWaves][kTieRows][M::NREC];
    __shared__ uint32_t thr_q[kWaves][PER ? 1 : 2 * kThrS];
    // opts: bit 0 = falling wave priorities; bits 8-15 = records the tie
    // queue may hold (as in the sc pass).
    const uint32_t prio = opts & 1u;
    const uint32_t b = xcd_block(blockIdx.x, grid);
    const ChainDev& C = pass_chain(chains, block_chain, b, total_blocks, opts, chain_m);
    const PassHead h = pass_head(C, b, total_blocks, s);
    const __amdgpu_buffer_rsrc_t ro = plane_rsrc(arena + h.off[A ^ 1u], h.plane);
    const __amdgpu_buffer_rsrc_t own = plane_rsrc(arena + h.off[A], h.plane);
    uint32_t (*const q_wave)[M::NREC] = tie_q[threadIdx.x >> 6];
    uint32_t* const thr_wave = thr_q[threadIdx.x >> 6];
    M m(C, h, opts, A, A == 1);
    m.load_thresholds(thr_wave);
    if (h.go) {
        const uint32_t ly = h.ly, lz = h.lz, w = h.w, pitch = h.pitch, y = h.y;
        const uint32_t z0 = h.zc * K, nk = min(K, lz - z0);
        const uint32_t i0 = m.i0, nvalid = m.nvalid, vmask = m.vmask;
        const bool px = PER || (h.pbc & 1u), py = PER || (h.pbc & 2u), pz = PER || (h.pbc & 4u);
        // y' = y - 1 (colour 0) or y + 1 (colour 1), wrapping when periodic
        const bool yok = (A == 0 ? y > 0 : y + 1 < ly) || py;
        const uint32_t dy = A == 0 ? (y > 0 ? 0u - pitch : (ly - 1) * pitch)
                                   : (y + 1 < ly ? pitch : 0u - (ly - 1) * pitch);
        // The x-offset position outside the segment: i0-1, or w-1 across the
        // periodic end (colour 0), or i0+32, or position 0 (colour 1), which
        // lands in the bit of the last valid position.  xe: the one site
        // whose x-offset neighbours are absent (open x; 32: none).
        const bool xr_in = i0 + kIsingSeg < w;
        const XPos xp = xpos(A == 0 ? (i0 > 0 ? i0 - 1 : w - 1)
                                           : (xr_in ? i0 + kIsingSeg : 0u));
        const bool xok = (A == 0 ? i0 > 0 : xr_in) || px;
        const uint32_t xe = xok ? 32u : (A == 0 ? 0u : nvalid - 1u);
        const uint32_t xr_sh = xr_in ? 31u : nvalid - 1u;
        const uint32_t woff = i0 >> 3;
        const uint32_t zstep = ly * pitch;

        // A pair as loaded: rows (y, zz) at rowoff and (y', zz).
        struct Pair {
            uint32_t r0, r1;
            uint32_t e0, e1;
        };
        const auto load_pair = [&](uint32_t rowoff, bool zok) {
            const uint32_t off1 = rowoff + dy;
            Pair p;
            p.r0 = load_word(ro, zok ? rowoff + woff : kNoRow);
            p.r1 = load_word(ro, zok && yok ? off1 + woff : kNoRow);
            p.e0 = load_word(ro, zok && xok ? rowoff + xp.off : kNoRow);
            p.e1 = load_word(ro, zok && yok && xok ? off1 + xp.off : kNoRow);
            return p;
        };
        // The word of the x-offset neighbours of a row.
        const auto shifted = [&](uint32_t r, uint32_t e) {
            const uint32_t bit = (e >> xp.sh) & 1u;
            return A == 0 ? (r << 1) | bit : (r >> 1) | (bit << xr_sh);
        };
        // Up neighbours 0..4 of the pair's rows.
        const auto count_pair = [&](const Pair& p, uint32_t c[3]) {
            const uint32_t r0 = arrived(p.r0) & vmask, r1 = arrived(p.r1) & vmask;
            const uint32_t s0 = shifted(r0, arrived(p.e0)), s1 = shifted(r1, arrived(p.e1));
            const uint32_t sum = bop3<kXor3>(r0, r1, s0), car = bop3<kMaj3>(r0, r1, s0);
            const uint32_t c2 = sum & s1;
            c[0] = sum ^ s1;
            c[1] = car ^ c2;
            c[2] = car & c2;
        };
        uint32_t row = y + ly * z0;
        uint32_t rowoff = row * pitch;
        // The lower pair of the first plane: zl = z0-1 (colour 0) or z0.
        bool lo_ok = A == 0 ? z0 > 0 || pz : true;
        uint32_t lo[3];
        count_pair(load_pair(A == 0 ? (z0 > 0 ? rowoff - zstep : rowoff + (lz - 1) * zstep) : rowoff,
                             lo_ok),
                   lo);
        const uint32_t wA = ctr_w(h.t, kIsingA, A);
        // The upper pair of plane z, zu = z (colour 0) or z+1 (colour 1), and
        // the own word as loaded; loads of the march's next plane are in
        // flight while a plane is decided.
        struct Plane {
            Pair hi;
            uint32_t own;
        };
        const auto load_plane = [&](uint32_t z, uint32_t roff, bool in) {
            const bool top = A == 1 && z + 1 == lz;
            const uint32_t hi_off = A == 0 ? roff : (top ? y * pitch : roff + zstep);
            Plane p;
            p.hi = load_pair(hi_off, in && (!top || pz));
            p.own = load_word(own, in ? roff + woff : kNoRow);
            return p;
        };
        Plane next = load_plane(z0, rowoff, true);
        const auto plane = [&](auto plain, uint32_t k) {
            constexpr bool PLAIN = decltype(plain)::value;
            // Falling priority while every wave is resident (as in the sc pass).
            if (prio) set_prio(((K - 1u - k) * 4u) / K);
            const uint32_t z = z0 + k;
            const bool hi_ok = !(A == 1 && z + 1 == lz) || pz;
            const Plane cur = next;
            if (k + 1 < K) next = load_plane(z + 1, rowoff + zstep, k + 1 < nk);
            Edge ed{0u, 0u, 32u, 0u, 0u};
            // present rows of the four, each with two slots (one at xe)
            const uint32_t nr = (lo_ok ? (yok ? 2u : 1u) : 0u) + (hi_ok ? (yok ? 2u : 1u) : 0u);
            if constexpr (!PER) ed = Edge{8u - 2u * nr, nr, xe, 0u, 0u};
            const uint32_t gw = m.template wave_absent<PLAIN>(ed);
            // draws first: they do not wait for the loads
            const U4 r0 = philox(U4{i0 >> 4, row, (uint32_t)h.t, wA}, h.k0, h.k1);
            const U4 r1 = philox(U4{(i0 >> 4) + 1u, row, (uint32_t)h.t, wA}, h.k0, h.k1);
            uint32_t d[8];
            draw_planes(r0, r1, d);
            keep_draws(d);
            const uint32_t o = arrived(cur.own);
            uint32_t hi[3], u[4], a[4];
            count_pair(cur.hi, hi);
            add_quads(lo, hi, u);
            if (gw == 0u)
                align_all<8>(u, o, a);
            else
                align_present(u, o, 2u * nr, nr, xe < 32u ? 1u << xe : 0u, a);
            m.template word<PLAIN>(own, q_wave, thr_wave, gw, o, a, nullptr, d, ed, rowoff + woff, row);
            lo[0] = hi[0];
            lo[1] = hi[1];
            lo[2] = hi[2];
            lo_ok = hi_ok;
            row += ly;
            rowoff += zstep;
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
    m.partials(partials, (uint64_t)(s * 2u + A) * total_blocks + b, h.active);
}

#define VG_BCC_PASS(A, K, MODE)                                                              \
    template __global__ void ising_bcc_pass<A, K, MODE>(const ChainDev*, const uint32_t*,    \
                                                        uint8_t*, int32_t*, uint32_t, uint32_t, \
                                                        uint32_t, uint32_t, uint32_t);
#define VG_BCC_COLOUR(A)         \
    VG_BCC_PASS(A, 1, kOpen)     \
    VG_BCC_PASS(A, 2, kOpen)     \
    VG_BCC_PASS(A, 4, kOpen)     \
    VG_BCC_PASS(A, 8, kOpen)     \
    VG_BCC_PASS(A, 1, kPeriodic) \
    VG_BCC_PASS(A, 2, kPeriodic) \
    VG_BCC_PASS(A, 4, kPeriodic) \
    VG_BCC_PASS(A, 8, kPeriodic)
VG_BCC_COLOUR(0)
VG_BCC_COLOUR(1)
#undef VG_BCC_COLOUR
#undef VG_BCC_PASS

}  // namespace vg
