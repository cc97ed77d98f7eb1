// fp32 Heisenberg checkerboard colour pass on the body-centred cubic
// lattice, for any number of chains packed in one arena.
//
// The per-site update is the one of the sc pass (heis_common.hpp); only the
// neighbour sum differs.  A corner site of cell (x,y,z) (colour 0) bonds to
// the body centres of cells (x-dx, y-dy, z-dz), a body centre (colour 1) to
// the corners of cells (x+dx, y+dy, z+dz), dx,dy,dz in {0,1}; the field h is
// summed over the eight slots in the order dz, dy, dx (dx fastest) with an
// absent slot (open boundary) adding +0.0f.
//
// Work item: S = 1 or 4 consecutive positions of one row; each of the four
// neighbour rows is read at the item's positions (with four, one aligned 16-byte
// load per component) and at the one position beyond it (x-1 or x+S).  Same
// three phases as the sc pass (fields and first proposal calls, the wave's
// queue, updates).
#include "heis_common.hpp"

namespace vg {

template <uint32_t S>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void heis_bcc_pass(const ChainDev* __restrict__ chains,
                                                     const uint32_t* __restrict__ block_chain,
                                                     float* __restrict__ arena,
                                                     int64_t* __restrict__ partials,
                                                     uint32_t colour, uint32_t s,
                                                     uint32_t total_blocks, uint32_t grid) {
    __shared__ HeisQueue hq[kBlock / 64];
    const uint32_t b = xcd_block(blockIdx.x, grid);
    const ChainDev& C = chains[block_chain[min(b, total_blocks - 1u)]];
    const HeisHead H = heis_head(C, b, total_blocks, s);
    if (!H.run) return;  // uniform: the workgroup belongs to one chain
    const bool active = H.active, rnd = H.proposal != 0;
    const uint64_t t = H.t;
    int32_t s32[4] = {0, 0, 0, 0};     // mx, my, mz, axis2 of the lane's sites
    int64_t bsum = 0;                  // bond of the lane's sites

    // Phase 1: neighbour fields, old spins and proposals of the item's sites.
    // Component planes through buffer resources: 32-bit byte offsets (a
    // component plane is below 4 GiB, checked on the host), and kNoRow reads
    // 0 for an absent neighbour row.
    __amdgpu_buffer_rsrc_t rown[3], roth[3];
    {
        const uint64_t plane = H.plane;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            rown[c] = plane_rsrc(reinterpret_cast<const uint8_t*>(arena + (colour ? H.off[1] : H.off[0]) + c * plane),
                                 (uint32_t)(plane * 4u));
            roth[c] = plane_rsrc(
                reinterpret_cast<const uint8_t*>(arena + (colour ? H.off[0] : H.off[1]) + c * plane),
                (uint32_t)(plane * 4u));
        }
    }
    // Every lane runs the same code: a lane past the chain's items (the
    // tail of its last block) has no valid site and its own row offset is
    // kNoRow, so it reads zeros and its stores are dropped; a site j >=
    // nvalid of a short last segment is padding, which every kernel keeps at
    // zero.  Neither is ever accepted, so both add zero to the sums.
    const uint32_t ly = H.ly, lz = H.lz, w = H.w, pitch = H.pitch, pbc = H.pbc;
    const uint32_t row = H.row;
    const uint32_t seg = H.seg;
    const uint32_t z = H.z, y = H.y;
    const bool px = pbc & 1u, py = pbc & 2u, pz = pbc & 4u;
    const uint32_t i0 = seg * S;
    const uint32_t nvalid = active ? min(S, w - i0) : 0u;
    const uint32_t own_off = active ? (row * pitch + i0) * 4u : kNoRow;
    uint32_t pend = 0;
    float os[S][3], hs[S][3], ps[S][3], us[S];
    {
        bool yok, zok;
        uint32_t y2, z2;
        if (colour == 0) {
            yok = y > 0 || py;
            y2 = y > 0 ? y - 1 : ly - 1;
            zok = z > 0 || pz;
            z2 = z > 0 ? z - 1 : lz - 1;
        } else {
            yok = y + 1 < ly || py;
            y2 = y + 1 < ly ? y + 1 : 0;
            zok = z + 1 < lz || pz;
            z2 = z + 1 < lz ? z + 1 : 0;
        }
        // slot rows in order (dy, dz) = (0,0), (1,0), (0,1), (1,1)
        const uint32_t rows[4] = {row, y2 + ly * z, y + ly * z2, y2 + ly * z2};
        const bool rok[4] = {true, yok, zok, yok && zok};
        // x offset of the second slot of each row: x-1 (colour 0), x+1 (colour 1)
        bool xe_ok;
        uint32_t xe_pos;
        if (colour == 0) {
            xe_pos = i0 > 0 ? i0 - 1 : w - 1;
            xe_ok = i0 > 0 || px;
        } else {
            xe_pos = i0 + S < w ? i0 + S : 0;
            xe_ok = i0 + S < w || px;
        }

        Run<S> so[3], v[4][3];
        // colour 1: the last segment's extra position is 0, the +x slot of
        // position w-1 across the periodic end (0 when x is open)
        float xe[4][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) so[c] = bload<S>(rown[c], own_off);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t ro = rows[r] * pitch * 4u;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v[r][c] = bload<S>(roth[c], rok[r] ? ro + i0 * 4u : kNoRow);
                xe[r][c] = bload1f(roth[c], rok[r] && xe_ok ? ro + xe_pos * 4u : kNoRow);
            }
        }

        heis_propose<S>(H.seed, rnd, colour, i0, row, t, us, ps, pend);
#pragma unroll
        for (uint32_t j = 0; j < S; ++j) {
#pragma unroll
            for (int c = 0; c < 3; ++c) os[j][c] = so[c].v[j];
            const uint32_t pos = i0 + j;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                float acc_h = 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float a = v[r][c].v[j];
                    float bx;
                    if (colour == 0)
                        bx = j == 0 ? xe[r][c] : v[r][c].v[j - 1];
                    else
                        bx = (pos + 1 == w || j == S - 1) ? xe[r][c] : v[r][c].v[j + 1];
                    acc_h = r == 0 ? fa(a, bx) : fa(fa(acc_h, a), bx);
                }
                hs[j][c] = acc_h;
            }
        }
        pend &= (1u << nvalid) - 1u;  // no further calls for sites that do not exist
    }

    // Phase 2: the wave's sites whose first proposal call missed.
    if (rnd) heis_resolve(H.seed, hq[threadIdx.x >> 6], pend, i0, row, t, colour, ps);

    // Phase 3: accept or reject, store, sums.
    {
        float ns[3][S];
#pragma unroll
        for (uint32_t j = 0; j < S; ++j) {
            float n[3];
            if (!rnd) {
#pragma unroll
                for (int c = 0; c < 3; ++c) ps[j][c] = -os[j][c];
            }
            heis_update(C, colour == 1, os[j], hs[j], hs[j], us[j], ps[j], n, s32, bsum,
                        j < nvalid);
            ns[0][j] = n[0];
            ns[1][j] = n[1];
            ns[2][j] = n[2];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            bstore<S>(rown[c], own_off, ns[c]);
        }
    }

    heis_partials_sites(s32, bsum, partials, colour, 2u, s, total_blocks, b);
}

#define VG_HEIS_BCC(S)                                                                \
    template __global__ void heis_bcc_pass<S>(const ChainDev*, const uint32_t*, float*, \
                                              int64_t*, uint32_t, uint32_t, uint32_t,   \
                                              uint32_t);
VG_HEIS_BCC(1)
VG_HEIS_BCC(4)
#undef VG_HEIS_BCC

}  // namespace vg
