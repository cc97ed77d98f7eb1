// Neighbours of the resident kernels, which hold a small chain's spins in LDS:
// site (colour c, row y + ly * z, position i) at index c * nc + row * w + i, nc
// sites a colour.
#pragma once

#include "fcc_common.hpp"

namespace vg {

// Index of the d-th neighbour slot of the colour-c site (y, z, i), in the order
// the passes sum them (of the two x slots of sc, whichever first), or `absent`
// past an open end.
template <uint32_t Z>
__device__ __forceinline__ uint32_t neighbour_at(const ChainDev& C, uint32_t c, uint32_t y,
                                                 uint32_t z, uint32_t i, uint32_t d, uint32_t nc,
                                                 uint32_t absent) {
    const bool px = C.pbc & 1u, py = C.pbc & 2u, pz = C.pbc & 4u;
    bool okx = true, oky = true, okz = true;
    uint32_t b = c ^ 1u;
    if constexpr (Z == 6) {
        if (d == 1u) i = fcc_move(i, ((c + y + z) & 1u) ? 1 : -1, C.w, px, okx);
        if (d == 2u || d == 3u) y = fcc_move(y, d == 2u ? -1 : 1, C.ly, py, oky);
        if (d >= 4u) z = fcc_move(z, d == 4u ? -1 : 1, C.lz, pz, okz);
    } else if constexpr (Z == 8) {
        const int st = c ? 1 : -1;
        if (d & 1u) i = fcc_move(i, st, C.w, px, okx);
        if (d & 2u) y = fcc_move(y, st, C.ly, py, oky);
        if (d & 4u) z = fcc_move(z, st, C.lz, pz, okz);
    } else {
        b = d >> 2;
        if (b >= c) ++b;
        const uint32_t axes = fcc_diff(c, b);
        // d's two bits along the two axes of the pair
        const bool first = d & 1u, second = d & 2u;
        const bool mx = (axes & 1u) && first;
        const bool my = (axes & 2u) && ((axes & 1u) ? second : first);
        const bool mz = (axes & 4u) && second;
        if (mx) i = fcc_move(i, fcc_step(c, b, 0), C.w, px, okx);
        if (my) y = fcc_move(y, fcc_step(c, b, 1), C.ly, py, oky);
        if (mz) z = fcc_move(z, fcc_step(c, b, 2), C.lz, pz, okz);
    }
    return okx && oky && okz ? b * nc + (y + C.ly * z) * C.w + i : absent;
}

}  // namespace vg
