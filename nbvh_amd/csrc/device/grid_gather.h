// grid_gather.h -- corner entries of hash-grid levels for the gathers of the matrix-core kernels.
#pragma once

#include "common.h"

namespace nbvh {
namespace dev {

// Entries (within the level) of the 8 corners of one level at point (x, y, z), and the fractional
// position. HASHED: the level is hashed (a power-of-two size), so only the coherent prime hash is
// formed: two multiplies per level, then one xor-and per corner. The hash of any position is in
// range, so this form is exact for points outside the unit cube too. Otherwise the general form
// (dense or hashed at run time, grid_corners) with its EXACT modulo switch.
template <bool HASHED, bool EXACT>
__device__ __forceinline__ void level_entries(const GridLevel& lv, float x, float y, float z, uint32_t idx[8],
                                              float fr[3])
{
    uint32_t g[3];
    grid_cell(lv, x, y, z, g, fr);
    if constexpr (HASHED) {
        const uint32_t hy0 = g[1] * 2654435761u, hy1 = hy0 + 2654435761u;
        const uint32_t hz0 = g[2] * 805459861u, hz1 = hz0 + 805459861u;
        const uint32_t yz[4] = {hy0 ^ hz0, hy1 ^ hz0, hy0 ^ hz1, hy1 ^ hz1};
        const uint32_t mask = lv.size - 1u, x1 = g[0] + 1u;
#pragma unroll
        for (int c = 0; c < 8; c++) idx[c] = (((c & 1) ? x1 : g[0]) ^ yz[c >> 1]) & mask;
    } else {
        grid_corners<EXACT>(lv, g, idx);
    }
}

// tcnn's weight of corner c, ((1 * w_x) * w_y) * w_z, from the fractional position.
__device__ __forceinline__ float trilinear_weight(int c, const float wx[2], const float wy[2], const float wz[2])
{
    return (wx[c & 1] * wy[(c >> 1) & 1]) * wz[c >> 2];
}

}  // namespace dev
}  // namespace nbvh
