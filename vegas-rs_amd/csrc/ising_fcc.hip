// Ising colour pass on the face-centred cubic lattice, multispin coded, for
// any number of chains packed in one arena.
//
// The same update as the sc and bcc passes (MetropolisFlipIntegrator::step /
// MetropolisIntegrator::step, reference src/integrator.rs:66-138, with the
// Exchange + Zeeman local energy of src/energy.rs:147-151, 194-206) on the
// fcc topology of Lattice::fcc (src/input.rs:296-322), which is not
// bipartite: a sweep is four passes, one per sublattice (fcc_common.hpp), each
// reading the three other planes.
//
// Work item: one 32-position segment of a row, marched up through K (the
// tile) consecutive z planes.  A sublattice A differs from each other one, b,
// along two axes, and bonds to four sites of it:
//   y, z: the rows (y, z), (y', z), (y, z'), (y', z') at x;
//   x, z: the rows (y, z), (y, z'), each at x and at the x offset;
//   x, y: the rows (y, z), (y', z), each at x and at the x offset
// (the offset: x-1 for colours 0 and 1, x+1 for colours 2 and 3).  With z' =
// z - 1 or z + 1 fixed per pair, the counts (0..2) of plane z' or z that the
// next plane needs again are kept, so a plane loads its own word, five of the
// others and the three that hold their x neighbour outside the segment.
// Counts and decision work on whole words (ising_word.hpp).  The pass of
// colour A adds the bonds to the lower colours b < A, so over a sweep every
// bond counts once.
#include "fcc_common.hpp"
#include "ising_word.hpp"

#include <type_traits>

namespace vg {

// The sublattice that differs from A along the axes `diff`.
__host__ __device__ constexpr uint32_t fcc_other(uint32_t a, uint32_t diff) {
    return fcc_diff(a, 0) == diff ? 0u : (fcc_diff(a, 1) == diff ? 1u : (fcc_diff(a, 2) == diff ? 2u : 3u));
}

template <uint32_t A, uint32_t K, uint32_t MODE>
__global__ __launch_bounds__(256) void ising_fcc_pass(const ChainDev* __restrict__ chains,
                                                      const uint32_t* __restrict__ block_chain,
                                                      uint8_t* __restrict__ arena,
                                                      int32_t* __restrict__ partials, uint32_t s,
                                                      uint32_t total_blocks, uint32_t grid,
                                                      uint32_t opts, uint32_t chain_m) {
    using M = March<12, A == 0 ? 0 : 2, MODE>;
    constexpr bool PER = M::PER;
    __shared__ uint32_t tie_q[kWaves][kTieRows][M::NREC];
    __shared__ uint32_t thr_q[kWaves][PER ? 1 : 2 * kThrS];
    // opts: bit 0 = falling wave priorities; bits 8-15 = records the tie
    // queue may hold (as in the sc pass).
    const uint32_t prio = opts & 1u;
    const uint32_t b = xcd_block(blockIdx.x, grid);
    const ChainDev& C = pass_chain(chains, block_chain, b, total_blocks, opts, chain_m);
    const PassHead h = pass_head(C, b, total_blocks, s);
    // the other sublattices by the axes they differ along
    constexpr uint32_t YZ = fcc_other(A, 6), XZ = fcc_other(A, 5), XY = fcc_other(A, 3);
    const __amdgpu_buffer_rsrc_t r_yz = plane_rsrc(arena + h.off[YZ], h.plane);
    const __amdgpu_buffer_rsrc_t r_xz = plane_rsrc(arena + h.off[XZ], h.plane);
    const __amdgpu_buffer_rsrc_t r_xy = plane_rsrc(arena + h.off[XY], h.plane);
    const __amdgpu_buffer_rsrc_t own = plane_rsrc(arena + h.off[A], h.plane);
    uint32_t (*const q_wave)[M::NREC] = tie_q[threadIdx.x >> 6];
    uint32_t* const thr_wave = thr_q[threadIdx.x >> 6];
    M m(C, h, opts, A, A > 0);
    m.load_thresholds(thr_wave);
    if (h.go) {
        const uint32_t ly = h.ly, lz = h.lz, w = h.w, pitch = h.pitch, y = h.y;
        const uint32_t z0 = h.zc * K, nk = min(K, lz - z0);
        const uint32_t i0 = m.i0, nvalid = m.nvalid, vmask = m.vmask;
        const bool px = PER || (h.pbc & 1u), py = PER || (h.pbc & 2u), pz = PER || (h.pbc & 4u);
        // row y' of the y, z and x, y pairs, relative to row y
        const auto ystep = [&](int d, bool& ok) {
            const uint32_t y2 = fcc_move(y, d, ly, py, ok);
            return (y2 - y) * pitch;
        };
        bool ok_yz, ok_xy;
        const uint32_t dy_yz = ystep(fcc_step(A, YZ, 1), ok_yz);
        const uint32_t dy_xy = ystep(fcc_step(A, XY, 1), ok_xy);
        if constexpr (PER) ok_yz = ok_xy = true;
        // The x-offset neighbour outside the segment: position i0-1 (colours
        // 0, 1) or i0+32, or position 0 across the periodic end (colours 2,
        // 3), which lands in the bit of the last valid position.  xe: the one
        // site whose x-offset neighbours are absent (open x; 32: none).
        constexpr bool kXneg = A < 2;
        const bool xr_in = i0 + kIsingSeg < w;
        const XPos xp = xpos(kXneg ? (i0 > 0 ? i0 - 1 : w - 1)
                                          : (xr_in ? i0 + kIsingSeg : 0u));
        const bool xok = (kXneg ? i0 > 0 : xr_in) || px;
        const uint32_t xe = xok ? 32u : (kXneg ? 0u : nvalid - 1u);
        const uint32_t xr_sh = xr_in ? 31u : nvalid - 1u;
        const uint32_t woff = i0 >> 3;
        const uint32_t zstep = ly * pitch;
        const auto word = [&](__amdgpu_buffer_rsrc_t r, uint32_t off, bool ok) {
            return load_word(r, ok ? off + woff : kNoRow);
        };
        const auto xword = [&](__amdgpu_buffer_rsrc_t r, uint32_t off, bool ok) {
            return load_word(r, ok && xok ? off + xp.off : kNoRow);
        };
        // The word of the x-offset neighbours of a row.
        const auto shifted = [&](uint32_t r, uint32_t e) {
            const uint32_t bit = (e >> xp.sh) & 1u;
            return kXneg ? (r << 1) | bit : (r >> 1) | (bit << xr_sh);
        };
        uint32_t row = y + ly * z0;
        uint32_t rowoff = row * pitch;
        // A pair that differs along z needs planes z and z' = z + sz; the
        // lower of the two is the upper of the plane before.  Both pairs of a
        // sublattice step the same way along z.
        constexpr int kSz = fcc_step(A, YZ, 2);
        static_assert(kSz == fcc_step(A, XZ, 2), "z steps of the two z pairs");
        bool lo_ok = kSz < 0 ? z0 > 0 || pz : true;
        const uint32_t lo_off =
            kSz < 0 ? (z0 > 0 ? rowoff - zstep : rowoff + (lz - 1) * zstep) : rowoff;
        uint32_t lyz[2], lxz[2];  // counts 0..2 of the lower plane
        {
            const uint32_t r0 = word(r_yz, lo_off, lo_ok);
            const uint32_t r1 = word(r_yz, lo_off + dy_yz, lo_ok && ok_yz);
            const uint32_t r2 = word(r_xz, lo_off, lo_ok) & vmask;
            const uint32_t x2 = shifted(r2, xword(r_xz, lo_off, lo_ok));
            lyz[0] = r0 ^ r1;
            lyz[1] = r0 & r1;
            lxz[0] = r2 ^ x2;
            lxz[1] = r2 & x2;
        }
        const uint32_t wA = ctr_w(h.t, kIsingA, A);
        // A plane's words as loaded, the z pairs' upper plane being z (step
        // -1) or z+1 (step +1); loads of the march's next plane are in flight
        // while a plane is decided.
        struct Plane {
            uint32_t own, yz0, yz1, xz, xy0, xy1;
            uint32_t e_xz, e_xy0, e_xy1;
        };
        const auto load_plane = [&](uint32_t z, uint32_t roff, bool in) {
            const bool top = kSz > 0 && z + 1 == lz;
            const bool hi = in && (!top || pz);
            const uint32_t hi_off = kSz < 0 ? roff : (top ? y * pitch : roff + zstep);
            Plane p;
            p.own = load_word(own, in ? roff + woff : kNoRow);
            p.yz0 = word(r_yz, hi_off, hi);
            p.yz1 = word(r_yz, hi_off + dy_yz, hi && ok_yz);
            p.xz = word(r_xz, hi_off, hi);
            p.e_xz = xword(r_xz, hi_off, hi);
            p.xy0 = word(r_xy, roff, in);
            p.xy1 = word(r_xy, roff + dy_xy, in && ok_xy);
            p.e_xy0 = xword(r_xy, roff, in);
            p.e_xy1 = xword(r_xy, roff + dy_xy, in && ok_xy);
            return p;
        };
        Plane next = load_plane(z0, rowoff, true);
        const auto plane = [&](auto plain, uint32_t k) {
            constexpr bool PLAIN = decltype(plain)::value;
            // Falling priority while every wave is resident (as in the sc pass).
            if (prio) set_prio(((K - 1u - k) * 4u) / K);
            const bool hi_ok = !(kSz > 0 && z0 + k + 1 == lz) || pz;
            const Plane cur = next;
            if (k + 1 < K) next = load_plane(z0 + k + 1, rowoff + zstep, k + 1 < nk);
            Edge ed{0u, 0u, 32u, 4u * A, 0u};
            uint32_t pres = 12u, miss = 0u;
            if constexpr (!PER) {
                // present slots of each pair at every site, and those of them
                // that are missing at xe
                const uint32_t nz = (lo_ok ? 1u : 0u) + (hi_ok ? 1u : 0u);
                uint32_t pr[4] = {0, 0, 0, 0}, ms[4] = {0, 0, 0, 0};
                pr[YZ] = nz * (ok_yz ? 2u : 1u);
                pr[XZ] = 2u * nz;
                ms[XZ] = nz;
                ms[XY] = ok_xy ? 2u : 1u;
                pr[XY] = 2u * ms[XY];
                pres = 0;
                uint32_t pl = 0, me = 0;
#pragma unroll
                for (uint32_t ob = 0; ob < 4; ++ob) {
                    pres += pr[ob];
                    miss += ms[ob];
                    if (ob < A) {
                        pl += pr[ob];
                        me += ms[ob];
                    }
                }
                ed = Edge{12u - pres, miss, xe, pl, me};
            }
            const uint32_t gw = m.template wave_absent<PLAIN>(ed);
            // draws first: they do not wait for the loads
            const U4 d0 = philox(U4{i0 >> 4, row, (uint32_t)h.t, wA}, h.k0, h.k1);
            const U4 d1 = philox(U4{(i0 >> 4) + 1u, row, (uint32_t)h.t, wA}, h.k0, h.k1);
            uint32_t d[8];
            draw_planes(d0, d1, d);
            keep_draws(d);

            const uint32_t o = arrived(cur.own);
            uint32_t qd[4][3];  // up neighbours 0..4 in each other sublattice
            {
                const uint32_t r0 = arrived(cur.yz0), r1 = arrived(cur.yz1);
                const uint32_t h0 = r0 ^ r1, h1 = r0 & r1;
                add_pairs(lyz[0], lyz[1], h0, h1, qd[YZ]);
                lyz[0] = h0;
                lyz[1] = h1;
            }
            {
                const uint32_t r = arrived(cur.xz) & vmask, x = shifted(r, arrived(cur.e_xz));
                const uint32_t h0 = r ^ x, h1 = r & x;
                add_pairs(lxz[0], lxz[1], h0, h1, qd[XZ]);
                lxz[0] = h0;
                lxz[1] = h1;
            }
            {
                const uint32_t r0 = arrived(cur.xy0) & vmask;
                const uint32_t r1 = arrived(cur.xy1) & vmask;
                const uint32_t x0 = shifted(r0, arrived(cur.e_xy0)), x1 = shifted(r1, arrived(cur.e_xy1));
                add_pairs(r0 ^ x0, r0 & x0, r1 ^ x1, r1 & x1, qd[XY]);
            }
            // 0..8 in the two lower other sublattices, then 0..12; l: the up
            // neighbours of colours below A
            constexpr uint32_t B0 = A == 0 ? 1u : 0u, B1 = A <= 1 ? 2u : 1u, B2 = A <= 2 ? 3u : 2u;
            uint32_t e8[4], u[4], a[4], l[4] = {0u, 0u, 0u, 0u};
            add_quads(qd[B0], qd[B1], e8);
            {
                const uint32_t k0 = e8[0] & qd[B2][0];
                u[0] = e8[0] ^ qd[B2][0];
                u[1] = bop3<kXor3>(e8[1], qd[B2][1], k0);
                const uint32_t k1 = bop3<kMaj3>(e8[1], qd[B2][1], k0);
                u[2] = bop3<kXor3>(e8[2], qd[B2][2], k1);
                u[3] = e8[3] ^ bop3<kMaj3>(e8[2], qd[B2][2], k1);
            }
            if constexpr (A == 1) {
                l[0] = qd[0][0];
                l[1] = qd[0][1];
                l[2] = qd[0][2];
            } else if constexpr (A > 1) {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) l[j] = A == 2 ? e8[j] : u[j];
            }
            if (gw == 0u)
                align_all<12>(u, o, a);
            else
                align_present(u, o, pres, pres - miss, xe < 32u ? 1u << xe : 0u, a);
            m.template word<PLAIN>(own, q_wave, thr_wave, gw, o, a, l, d, ed, rowoff + woff, row);
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
        m.fold(nk, 4u * A);
    }
    m.settle_queue(own, q_wave, h.pitch, 4u * A);
    m.partials(partials, (uint64_t)(s * 4u + A) * total_blocks + b, h.active);
}

#define VG_FCC_PASS(A, K, MODE)                                                              \
    template __global__ void ising_fcc_pass<A, K, MODE>(const ChainDev*, const uint32_t*,    \
                                                        uint8_t*, int32_t*, uint32_t, uint32_t, \
                                                        uint32_t, uint32_t, uint32_t);
#define VG_FCC_COLOUR(A)         \
    VG_FCC_PASS(A, 1, kOpen)     \
    VG_FCC_PASS(A, 2, kOpen)     \
    VG_FCC_PASS(A, 4, kOpen)     \
    VG_FCC_PASS(A, 8, kOpen)     \
    VG_FCC_PASS(A, 1, kPeriodic) \
    VG_FCC_PASS(A, 2, kPeriodic) \
    VG_FCC_PASS(A, 4, kPeriodic) \
    VG_FCC_PASS(A, 8, kPeriodic)
VG_FCC_COLOUR(0)
VG_FCC_COLOUR(1)
VG_FCC_COLOUR(2)
VG_FCC_COLOUR(3)
#undef VG_FCC_COLOUR
#undef VG_FCC_PASS

}  // namespace vg
