// mlp_f32.h -- the FP32 network on the FP32 matrix cores (v_mfma_f32_32x32x2_f32), 64 segments
// per wave, bit-identical to the scalar sequence acc = fmaf(W[j][k], x[k], acc), k ascending.
//
// v_mfma_f32_32x32x2_f32 adds its two products one after the other, each as a fused multiply-add
// rounded to FP32 (subnormals kept): 32 x 32 dot products of length 2 continue 32 x 32 fmaf
// chains. A layer is H_next^T = W * H^T, two blocks of 32 neurons x two blocks of 32 segments:
//   A (weights): lane l holds row l % 32, k = 2 s + l / 32 of k-step s;
//   B (activations): lane l holds segment l % 32, k = 2 s + l / 32;
//   D: lane l holds segment l % 32, rows 8 (r / 4) + 4 (l / 32) + r % 4 in register r.
// The host orders the weight rows of the hidden layers so that register r of row block rb is
// neuron 2 (16 rb + r) + l / 32: after the ReLU, register 16 rb + r IS the B operand of k-step
// 16 rb + r of the next layer, with k ascending (f32_fragments, host/mfma_layout.cpp).
// Layer 1: every lane gathers the K0 features of its own segment; one v_permlane32_swap per
// feature pair (2s, 2s+1) leaves the B operands of both segment blocks.
//
// What bounds it: with the gathers' lines in flight (two waves per SIMD, one gathering while the
// other multiplies) the random lines set the time, as in the FP16 kernel. The matrix cores give
// 256 FLOP per cycle and CU, twice the FMA rate without packed FP32, and leave the vector unit to
// the gathers' addresses: a wave's evaluation holds its matrix core for 41 k cycles (64 segments x
// 37,888 FLOP, the output layer padded from 8 to 32 rows). Measured, 1024 x 1024 camera rays of
// the benchmark object (1.4 M segments, 16 x 2 grid): 2957 us with the MLP as scalar FMAs at one
// wave per SIMD, 1870 us here; with the common level order (level_phases) and descended nodes kept,
// 2770 us there and 1601 us here, timed in turn.
#pragma once

#include "grid_gather.h"

namespace nbvh {
namespace dev {

typedef float floatx16_t __attribute__((ext_vector_type(16)));

// Weight fragments: layer 1, three hidden layers, output (floats). Within a layer two k-steps are
// paired per lane: ((rb * steps / 2 + s / 2) * 64 + lane) * 2 + s % 2. The output layer keeps its
// 8 rows only, ((s / 2 * 2 + l / 32) * 8 + row) * 2 + s % 2: rows 8..31 of its block repeat them.
template <int K0>
struct F32Layout {
    static constexpr int S1     = K0 / 2;
    static constexpr int HID    = 64 * K0;
    static constexpr int OUT    = HID + 3 * 64 * 64;
    static constexpr int FLOATS = OUT + 8 * 64;
    static_assert(K0 % 4 == 0, "k-steps come in pairs");
};

template <int K0>
__device__ __forceinline__ void stage_weights_f32(const float* __restrict__ frag, float4* lds)
{
    const float4* src = reinterpret_cast<const float4*>(frag);
    for (uint32_t i = threadIdx.x; i < (uint32_t)F32Layout<K0>::FLOATS / 4u; i += blockDim.x) lds[i] = src[i];
}

// Features of one level for all P points: all corner entries, then all loads, then the weights and
// the accumulation over corners 0..7. out[p * F + f].
template <int P, int F, bool HASHED, bool EXACT>
__device__ __forceinline__ void gather_level_f32(const GridLevel& lv, const float* __restrict__ tables,
                                                 const float* pts, float* out)
{
    typedef float entry_t __attribute__((ext_vector_type(F)));
    uint32_t idx[P][8];
    float fr[P][3];
#pragma unroll
    for (int p = 0; p < P; p++)
        level_entries<HASHED, EXACT>(lv, pts[3 * p], pts[3 * p + 1], pts[3 * p + 2], idx[p], fr[p]);
    // A uniform base per level and a 32-bit byte offset in it (2^26 entries of 16 bytes at most).
    const char* base = reinterpret_cast<const char*>(tables + (size_t)lv.offset * F);
    entry_t q[P][8];
#pragma unroll
    for (int p = 0; p < P; p++)
#pragma unroll
        for (int c = 0; c < 8; c++)
            q[p][c] = *reinterpret_cast<const entry_t*>(base + idx[p][c] * (uint32_t)sizeof(entry_t));
#pragma unroll
    for (int p = 0; p < P; p++) {
        const float wx[2] = {1.f - fr[p][0], fr[p][0]}, wy[2] = {1.f - fr[p][1], fr[p][1]};
        const float wz[2] = {1.f - fr[p][2], fr[p][2]};
#pragma unroll
        for (int k = 0; k < F; k++) out[p * F + k] = 0.f;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const float w = trilinear_weight(c, wx, wy, wz);
#pragma unroll
            for (int k = 0; k < F; k++) out[p * F + k] = fmaf(w, q[p][c][k], out[p * F + k]);
        }
    }
}

// All features, x[p * L * F + l * F + f]. ND >= 0: levels [ND, L) are hashed (n_dense == ND,
// checked at launch); ND < 0: any grid. G: the order of the levels.
template <int P, int L, int F, int ND, bool EXACT, Gather G>
__device__ __forceinline__ void gather_features_f32(const NetArgs& a, const float* __restrict__ tables,
                                                    const float* pts, float* x)
{
#pragma unroll
    for (int l = 0; l < (ND >= 0 ? ND : L); l++) {
        float r[P * F];
        gather_level_f32<P, F, false, EXACT>(a.level[l], tables, pts, r);
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int k = 0; k < F; k++) x[(p * L + l) * F + k] = r[p * F + k];
    }
    if constexpr (ND >= 0 && G == Gather::PHASES) {
        level_phases<L - ND>([&](uint32_t l) {
            float r[P * F];
            gather_level_f32<P, F, true, false>(a.level[ND + l], tables, pts, r);
#pragma unroll
            for (int i = 0; i < L - ND; i++)
#pragma unroll
                for (int p = 0; p < P; p++)
#pragma unroll
                    for (int k = 0; k < F; k++) {
                        float& w = x[(p * L + ND + i) * F + k];
                        w = l == (uint32_t)i ? r[p * F + k] : w;
                    }
        });
    } else if constexpr (ND >= 0) {
#pragma unroll
        for (int l = ND; l < L; l++) {
            float r[P * F];
            gather_level_f32<P, F, true, false>(a.level[l], tables, pts, r);
#pragma unroll
            for (int p = 0; p < P; p++)
#pragma unroll
                for (int k = 0; k < F; k++) x[(p * L + l) * F + k] = r[p * F + k];
        }
    }
}

// The features of this lane's own segment, every lane of the wave taking part.
template <int P, int L, int F, int ND, Gather G>
__device__ __forceinline__ void wave_features_f32(const NetArgs& a, const float* __restrict__ tables,
                                                  const float* pts, float* x)
{
#pragma unroll
    for (int k = 0; k < P * L * F; k++) x[k] = 0.f;
    if (__all(in_unit_cube<3 * P>(pts)))
        gather_features_f32<P, L, F, ND, false, G>(a, tables, pts, x);
    else
        gather_features_f32<P, L, F, ND, true, G>(a, tables, pts, x);
}

// WIDE gather of the wave's first `slots` slots (every lane takes part): round by round, lane =
// level * S + slot of S slots; then each of those slots' lanes collects its levels.
template <int P, int L, int F>
__device__ __forceinline__ void gather_wide_f32(const NetArgs& a, const float* __restrict__ tables, uint32_t slots,
                                                const float* pts, float* x)
{
    static_assert(64 % L == 0, "whole levels per wave");
    constexpr int S = 64 / L < 16 ? 64 / L : 16;
    const uint32_t lane = threadIdx.x & 63u;
    const GridLevel lv = a.level[lane / S < (uint32_t)L ? lane / S : 0];
#pragma unroll
    for (int k = 0; k < P * L * F; k++) x[k] = 0.f;
    for (uint32_t r = 0; r < slots; r += S) {
        float pt[3 * P], f[P * F];
#pragma unroll
        for (int c = 0; c < 3 * P; c++) pt[c] = __shfl(pts[c], (int)(r + lane % S));
        if (__all(in_unit_cube<3 * P>(pt)))
            gather_level_f32<P, F, false, false>(lv, tables, pt, f);
        else
            gather_level_f32<P, F, false, true>(lv, tables, pt, f);
        const bool mine = lane - r < (uint32_t)S;
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int l = 0; l < L; l++)
#pragma unroll
                for (int k = 0; k < F; k++) {
                    const float v = __shfl(f[p * F + k], (int)(l * S + lane % S));
                    float& w = x[(p * L + l) * F + k];
                    w = mine ? v : w;
                }
    }
}

// Own features -> B operands of layer 1: x[2s] serves segments 0..31, x[2s + 1] segments 32..63.
template <int K0>
__device__ __forceinline__ void features_to_b_f32(float* x)
{
#pragma unroll
    for (int s = 0; s < K0 / 2; s++) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[2 * s]), __float_as_uint(x[2 * s + 1]),
                                                        false, false);
        x[2 * s]     = __uint_as_float(r[0]);
        x[2 * s + 1] = __uint_as_float(r[1]);
    }
}

template <int CB>
__device__ __forceinline__ void zero_acc(floatx16_t acc[2][CB])
{
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[rb][cb][r] = 0.f;
}

// acc[rb][cb] += (row block rb of the S k-steps' weights) x (segment block cb): b[2 s + cb].
template <int S, int CB>
__device__ __forceinline__ void layer_f32(const float2* w, uint32_t lane, const float* b, floatx16_t acc[2][CB])
{
#pragma unroll
    for (int s = 0; s < S; s += 2) {
        const float2 w0 = w[(s / 2) * 64 + lane], w1 = w[(S / 2 + s / 2) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int cb = 0; cb < CB; cb++) {
                    const float wa = rb == 0 ? (e ? w0.y : w0.x) : (e ? w1.y : w1.x);
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa, b[2 * (s + e) + cb], acc[rb][cb], 0, 0, 0);
                }
    }
}

template <int CB>
__device__ __forceinline__ void relu_to_b_f32(const floatx16_t acc[2][CB], float b[64])
{
#pragma unroll
    for (int s = 0; s < 32; s++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const float v = acc[s / 16][cb][s % 16];
            b[2 * s + cb] = v > 0.f ? v : 0.f;
        }
}

// The MLP of the first 32 * CB segments of a wave. x[K0]: this lane's own features (overwritten);
// w: the weight fragments in LDS; z[8]: this lane's logits.
template <int K0, int CB>
__device__ __forceinline__ void mlp_wave_f32(const float* w, float* x, float z[8])
{
    typedef F32Layout<K0> Y;
    const uint32_t lane = threadIdx.x & 63u, g = lane >> 5;
    features_to_b_f32<K0>(x);
    floatx16_t acc[2][CB];
    zero_acc<CB>(acc);
    layer_f32<Y::S1, CB>(reinterpret_cast<const float2*>(w), lane, x, acc);
    float b[64];
#pragma unroll
    for (int layer = 0; layer < 3; layer++) {
        relu_to_b_f32<CB>(acc, b);
        zero_acc<CB>(acc);
        layer_f32<32, CB>(reinterpret_cast<const float2*>(w + Y::HID) + layer * 2048, lane, b, acc);
    }
    relu_to_b_f32<CB>(acc, b);
    floatx16_t out[2] = {};
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int r = 0; r < 16; r++) out[cb][r] = 0.f;
    const float2* wo = reinterpret_cast<const float2*>(w + Y::OUT);
#pragma unroll
    for (int s = 0; s < 32; s += 2) {
        const float2 v = wo[(s + g) * 8 + (lane & 7u)];
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
            for (int cb = 0; cb < CB; cb++)
                out[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(e ? v.y : v.x, b[2 * (s + e) + cb], out[cb], 0, 0, 0);
    }
    // Rows 0..3 of a segment block sit in lanes 0..31, rows 4..7 in lanes 32..63.
    float send[4], recv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        send[r] = g ? out[0][r] : out[1][r];
        recv[r] = __shfl_xor(send[r], 32);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        z[r]     = g ? recv[r] : out[0][r];
        z[4 + r] = g ? out[1][r] : recv[r];
    }
}

}  // namespace dev
}  // namespace nbvh
