// grid_gather.h -- corner entries of hash-grid levels for the gathers of the matrix-core kernels.
#pragma once

#include "common.h"

namespace nbvh {
namespace dev {

// Entries (within the level) of the 8 corners of cell g on a hashed level (a power-of-two size): the
// coherent prime hash alone, two multiplies per cell, then one xor-and per corner.
__device__ __forceinline__ void hash_corners(const GridLevel& lv, const uint32_t g[3], uint32_t idx[8])
{
    const uint32_t hy0 = g[1] * 2654435761u, hy1 = hy0 + 2654435761u;
    const uint32_t hz0 = g[2] * 805459861u, hz1 = hz0 + 805459861u;
    const uint32_t yz[4] = {hy0 ^ hz0, hy1 ^ hz0, hy0 ^ hz1, hy1 ^ hz1};
    const uint32_t mask = lv.size - 1u, x1 = g[0] + 1u;
#pragma unroll
    for (int c = 0; c < 8; c++) idx[c] = (((c & 1) ? x1 : g[0]) ^ yz[c >> 1]) & mask;
}

// Entries (within the level) of the 8 corners of one level at point (x, y, z), and the fractional
// position. HASHED: the level is hashed, so only hash_corners is formed. The hash of any position is
// in range, so this form is exact for points outside the unit cube too. Otherwise the general form
// (dense or hashed at run time, grid_corners) with its EXACT modulo switch.
template <bool HASHED, bool EXACT>
__device__ __forceinline__ void level_entries(const GridLevel& lv, float x, float y, float z, uint32_t idx[8],
                                              float fr[3])
{
    uint32_t g[3];
    grid_cell(lv, x, y, z, g, fr);
    if constexpr (HASHED) {
        hash_corners(lv, g, idx);
    } else {
        grid_corners<EXACT>(lv, g, idx);
    }
}

// tcnn's weight of corner c, ((1 * w_x) * w_y) * w_z, from the fractional position.
__device__ __forceinline__ float trilinear_weight(int c, const float wx[2], const float wy[2], const float wz[2])
{
    return (wx[c & 1] * wy[(c >> 1) & 1]) * wz[c >> 2];
}

// How a wave gathers the features of its slots.
//   LEVELS  every lane its own segment, level after level (the three points of a level together);
//   PAIRS   the same two levels at a time: twice the loads in flight, for launches with few waves;
//   PHASES  level by level, the hashed levels in the order of level_phases;
//   WIDE    few slots per wave: a lane takes one level of one slot, 64 / L slots at a time, so that
//           a segment costs one memory round trip instead of one per level.
enum class Gather { LEVELS, PHASES, WIDE, PAIRS };

// Visit each of N levels once, f(level) with a wave-uniform level, starting with the level whose
// turn it is: the turn moves every kLevelTicks of the 100 MHz clock, alike on every CU. The tables
// of all hashed levels (2 MB each at 2^19 entries in FP16, 12 of them) are six times an XCD's 4 MB
// L2, but one or two levels fit: waves that agree on the level share its lines there, and a wave
// that falls behind skips ahead to the common level and returns to the others later.
// Measured (us, gather order: all levels of a point / levels / phases): 1024 x 1024 camera rays
// 1300 / 1258 / 1164, 4M incoherent rays 13143 / 12311 / 11310, FP32 camera rays 1760 / - / 1690,
// 1M scattered segments in the network kernel, whose waves keep step by themselves, 2204 / 1685 /
// 1800 and more. Counters on the benchmark frame: L2 hits 43 -> 54 % of the requests, 32.2 -> 24.6 M
// lines missed, mean latency 471 -> 407 cycles. Ticks of 128 / 192 / 256 / 384 / 512: 1231 / 1179 / 1164 / 1170 / 1170 us.
constexpr uint32_t kLevelTicks = 256;
template <int N, typename Fn>
__device__ __forceinline__ void level_phases(const Fn& f)
{
    static_assert(N >= 1 && N < 32, "one bit per level");
    uint32_t left = (1u << N) - 1u;
#pragma clang loop unroll(disable)
    while (left != 0u) {
        const uint32_t turn = ((uint32_t)__builtin_amdgcn_s_memrealtime() / kLevelTicks) % (uint32_t)N;
        const uint32_t now  = (uint32_t)__builtin_amdgcn_readfirstlane((int)turn);
        const uint32_t up   = left >> now;
        const uint32_t l    = up != 0u ? now + (uint32_t)__builtin_ctz(up) : (uint32_t)__builtin_ctz(left);
        left &= ~(1u << l);
        f(l);
    }
}

// Grids of fewer hashed levels gain nothing from phases (8 levels, 4 of them hashed: 402 us either
// way on a 1013 x 691 frame: 8 MB of hashed tables, two levels to an L2 without any order, and 73 %
// of the requests hit there).
template <int L, int ND>
constexpr Gather kQueryGather = ND >= 0 && L - ND >= 8 ? Gather::PHASES : Gather::LEVELS;

// Next chunk of a persistent network kernel after the one at base < n, or n: base + step may pass 2^32
// for the last 2^32 - n < step inputs, and must not start again at the first ones.
__device__ __forceinline__ uint32_t next_chunk(uint32_t base, uint32_t group, uint32_t n)
{
    const uint32_t step = gridDim.x * group;
    return n - base > step ? base + step : n;
}

// The network kernels' waves keep step by themselves, so many hashed levels go one at a time; with
// few of them two at a time.
// Measured (1M scattered segments, us, levels / pairs): 8 x 4 grid FP16 704 / 683, FP8 731 / 679
// (all four levels of one point together: 695 / 713); 16 x 2 grid FP16 1678 / 1750, FP8 1735 / 1812.
template <int L, int ND>
constexpr Gather kNetworkGather = ND >= 0 && L - ND < 8 ? Gather::PAIRS : Gather::LEVELS;

}  // namespace dev
}  // namespace nbvh
