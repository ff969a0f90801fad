// neural_mfma.hip -- FP16 / BF16 / FP8 neural query and network inference on CDNA4 matrix cores.
//
// One wave evaluates 64 segments per iteration (the slots of the persistent wave scheduler):
//   * FP16 hash tables (scaled by a power of two), trilinear interpolation in FP32;
//   * the MLP as H^T = W * X^T with v_mfma_f32_32x32x16_{f16,bf16}: two 32-neuron row blocks x
//     two 32-segment column blocks per layer, FP32 accumulation, weights staged once per block
//     in LDS as ready-made A fragments (one ds_read_b128 per lane and MFMA);
//   * the accumulators of a layer become the B operand of the next after ReLU + conversion,
//     in registers (weights are pre-permuted on the host, host/mfma_layout.cpp);
//   * layer-1 B operands: each lane gathers the features of its own segment, one
//     v_permlane32_swap per register pair moves the halves into the operand layout.
#include <hip/hip_runtime.h>

#include "../device/grid_gather.h"
#include "../device/wave_query.h"
#include "launch.h"

namespace nbvh {
namespace dev {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

template <bool BF16>
struct Frag;
template <>
struct Frag<false> {
    typedef half8_t vec;
    typedef _Float16 elem;
    static __device__ __forceinline__ floatx16 mfma(vec a, vec b, floatx16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Frag<true> {
    typedef bf16x8_t vec;
    typedef __bf16 elem;
    static __device__ __forceinline__ floatx16 mfma(vec a, vec b, floatx16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

// Number of fragments for K0 inputs, 64 hidden, 4 hidden layers, 8 outputs.
template <int K0>
struct MlpShape {
    static constexpr int KS1    = K0 / 16;        // layer-1 k-steps
    static constexpr int F_L1   = 2 * KS1;        // layer-1 fragments
    static constexpr int F_HID  = 2 * 4;          // fragments per hidden layer
    static constexpr int N_FRAG = F_L1 + 3 * F_HID + 4;
};

// v_permlane32_swap(x, y): lanes 32..63 of x <-> lanes 0..31 of y, on 16-byte fragments.
template <typename V>
__device__ __forceinline__ void swap_halves(V& x, V& y)
{
    uint4 a = __builtin_bit_cast(uint4, x), b = __builtin_bit_cast(uint4, y);
    const auto r0 = __builtin_amdgcn_permlane32_swap(a.x, b.x, false, false);
    const auto r1 = __builtin_amdgcn_permlane32_swap(a.y, b.y, false, false);
    const auto r2 = __builtin_amdgcn_permlane32_swap(a.z, b.z, false, false);
    const auto r3 = __builtin_amdgcn_permlane32_swap(a.w, b.w, false, false);
    a = make_uint4(r0[0], r1[0], r2[0], r3[0]);
    b = make_uint4(r0[1], r1[1], r2[1], r3[1]);
    x = __builtin_bit_cast(V, a);
    y = __builtin_bit_cast(V, b);
}

template <int F>
__device__ __forceinline__ void load_corner(__amdgpu_buffer_rsrc_t tab, uint32_t off, uint32_t q[F / 2])
{
    if constexpr (F == 2) {
        q[0] = __builtin_amdgcn_raw_buffer_load_b32(tab, off, 0, 0);
    } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(tab, off, 0, 0);
        q[0] = v[0];
        q[1] = v[1];
    }
}

// Layer-1 B operands. Every lane computes all K0 features of its own segment (wave-uniform
// gather code); lo[s] holds features 8s..8s+7, hi[s] features K0/2+8s..K0/2+8s+7. Column block 0
// (segments 0..31) needs lo from lanes 0..31 and hi of the same segments in lanes 32..63;
// column block 1 (segments 32..63) needs lo of those segments in lanes 0..31 and hi in lanes
// 32..63. Swapping lanes 32..63 of lo with lanes 0..31 of hi (layer1_operands) produces exactly
// these operands, matching the weight order K(s, g, e) = g*K0/2 + 8s + e of host/mfma_layout.cpp.
//
// Features of all P points of this lane's segment, converted to 16 bits as each level completes:
// feature k = p*L*F + l*F + f goes to lo[k/8][k%8] (k < K0/2) or hi[(k-K0/2)/8][..]. The FP16
// tables are read through a buffer resource: 32-bit byte offsets (one VGPR per gather), and the
// hardware range check returns 0 for any offset past the table instead of faulting.
//
// Byte offsets of the 8 corners of one level at point (x, y, z) in the whole FP16 table, and the
// fractional position (level_entries: HASHED and EXACT).
template <int F, bool HASHED, bool EXACT>
__device__ __forceinline__ void level_offsets(const GridLevel& lv, float x, float y, float z, uint32_t off[8],
                                              float fr[3])
{
    constexpr uint32_t kShift = F == 2 ? 2u : 3u;  // log2 of the entry bytes (F halves)
    uint32_t idx[8];
    level_entries<HASHED, EXACT>(lv, x, y, z, idx, fr);
#pragma unroll
    for (int c = 0; c < 8; c++) off[c] = (idx[c] + lv.offset) << kShift;
}

// NL consecutive levels (lv[0 .. NL)), all P points: the corner offsets, then all 8 NL P loads, then
// the corner weights and the FP32 accumulation over corners 0..7 (tcnn's trilinear weights).
// out[(l * P + p) * F / 2 ..]: the features of point p at level l as 16-bit pairs.
template <int P, int F, bool BF16, bool HASHED, bool EXACT, int NL = 1>
__device__ __forceinline__ void gather_level(const GridLevel* lv, __amdgpu_buffer_rsrc_t tab, const float* points,
                                             uint32_t* out)
{
    constexpr int N = NL * P;
    typedef typename Frag<BF16>::elem E;
    typedef E pair_t __attribute__((ext_vector_type(2)));
    uint32_t off[N][8];
    float fr[N][3];
#pragma unroll
    for (int p = 0; p < N; p++)
    {
        const float* pt = points + 3 * (p % P);
        level_offsets<F, HASHED, EXACT>(lv[p / P], pt[0], pt[1], pt[2], off[p], fr[p]);
    }
    // One load per corner. (Measured: serving x-neighbour corners with one 16-byte load plus a
    // range-masked second load halves the throughput, so corners stay separate.)
    uint32_t q[N][8][F / 2];
#pragma unroll
    for (int p = 0; p < N; p++)
#pragma unroll
        for (int c = 0; c < 8; c++) load_corner<F>(tab, off[p][c], q[p][c]);
#pragma unroll
    for (int p = 0; p < N; p++) {
        // tcnn's corner weights ((1 * w_x) * w_y) * w_z, the x-y products shared by the z pair.
        const float wx[2] = {1.f - fr[p][0], fr[p][0]}, wy[2] = {1.f - fr[p][1], fr[p][1]};
        const float wz[2] = {1.f - fr[p][2], fr[p][2]};
        float acc[F];
#pragma unroll
        for (int k = 0; k < F; k++) acc[k] = 0.f;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const float w = trilinear_weight(c, wx, wy, wz);
#pragma unroll
            for (int k = 0; k < F; k++) {
                const uint32_t bits = (k & 1) ? (q[p][c][k / 2] >> 16) : (q[p][c][k / 2] & 0xFFFFu);
                acc[k] = fmaf(w, half_bits_to_float(bits), acc[k]);
            }
        }
#pragma unroll
        for (int j = 0; j < F / 2; j++) {
            const pair_t v = {(E)acc[2 * j], (E)acc[2 * j + 1]};
            out[p * (F / 2) + j] = __builtin_bit_cast(uint32_t, v);
        }
    }
}

// All features of the lane's segment, pair j of feature k = 2j, 2j + 1 (k = p * L * F + l * F + f).
// ND >= 0: the kernel is specialised for grids whose levels [ND, L) are hashed (n_dense == ND,
// checked at launch): those levels take the hash-only form, the others the general form. ND < 0:
// every level takes the general form (any grid). EXACT: the full modulo for points outside the
// unit cube (dense levels only; the hash is exact everywhere).
template <int P, int L, int F, bool BF16, bool EXACT, int ND, Gather G>
__device__ __forceinline__ void gather_operands(const NetArgs& a, __amdgpu_buffer_rsrc_t tab, const float* pts,
                                                uint32_t* x)
{
    static_assert(F == 2 || F == 4, "FP16 gather implemented for F = 2 and F = 4");
    constexpr int H = F / 2;  // 16-bit pairs per level and point
#pragma unroll
    for (int l = 0; l < (ND >= 0 ? ND : L); l++) {
        uint32_t r[P * H];
        gather_level<P, F, BF16, false, EXACT>(a.level + l, tab, pts, r);
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int j = 0; j < H; j++) x[(p * L + l) * H + j] = r[p * H + j];
    }
    if constexpr (ND >= 0) {
        if constexpr (G == Gather::PHASES) {
            level_phases<L - ND>([&](uint32_t l) {
                uint32_t r[P * H];
                gather_level<P, F, BF16, true, false>(a.level + ND + l, tab, pts, r);
#pragma unroll
                for (int i = 0; i < L - ND; i++)
#pragma unroll
                    for (int p = 0; p < P; p++)
#pragma unroll
                        for (int j = 0; j < H; j++) {
                            uint32_t& w = x[(p * L + ND + i) * H + j];
                            w = l == (uint32_t)i ? r[p * H + j] : w;
                        }
            });
        } else {
            constexpr int NL = G == Gather::PAIRS && (L - ND) % 2 == 0 ? 2 : 1;
#pragma unroll
            for (int l0 = ND; l0 < L; l0 += NL) {
                uint32_t r[NL * P * H];
                gather_level<P, F, BF16, true, false, NL>(a.level + l0, tab, pts, r);
#pragma unroll
                for (int l = 0; l < NL; l++)
#pragma unroll
                    for (int p = 0; p < P; p++)
#pragma unroll
                        for (int j = 0; j < H; j++) x[(p * L + l0 + l) * H + j] = r[(l * P + p) * H + j];
            }
        }
    }
}

// WIDE gather of the wave's first `slots` slots: round by round, lane = level * S + slot of 64 / L
// slots; then each of those slots' lanes collects its levels (one ds_bpermute per 16-bit pair).
template <int P, int L, int F, bool BF16>
__device__ __forceinline__ void gather_wide(const NetArgs& a, __amdgpu_buffer_rsrc_t tab, uint32_t slots,
                                            const float* pts, uint32_t* x)
{
    static_assert(64 % L == 0, "whole levels per wave");
    constexpr int S = 64 / L, H = F / 2;
    const uint32_t lane = threadIdx.x & 63u;
    const GridLevel lv = a.level[lane / S];
    for (uint32_t r = 0; r < slots; r += S) {
        float pt[3 * P];
#pragma unroll
        for (int c = 0; c < 3 * P; c++) pt[c] = __shfl(pts[c], (int)(r + lane % S));
        uint32_t f[P * H];
        if (__all(in_unit_cube<3 * P>(pt)))
            gather_level<P, F, BF16, false, false>(&lv, tab, pt, f);
        else
            gather_level<P, F, BF16, false, true>(&lv, tab, pt, f);
        const bool mine = lane - r < (uint32_t)S;
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int l = 0; l < L; l++)
#pragma unroll
                for (int j = 0; j < H; j++) {
                    const uint32_t v = (uint32_t)__shfl((int)f[p * H + j], (int)(l * S + lane % S));
                    uint32_t& w = x[(p * L + l) * H + j];
                    w = mine ? v : w;
                }
    }
}

template <int P, int L, int F, bool BF16, int ND, Gather G>
__device__ __forceinline__ void layer1_operands(const NetArgs& a, uint32_t slots, const float* pts,
                                                typename Frag<BF16>::vec lo[P * L * F / 16],
                                                typename Frag<BF16>::vec hi[P * L * F / 16])
{
    constexpr int K0 = P * L * F;
    typedef typename Frag<BF16>::vec V;
    const __amdgpu_buffer_rsrc_t tab =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.tables_f16, (short)0, (int)a.tables_f16_bytes, 0x00020000);
    uint32_t x[K0 / 2] = {};
    if constexpr (G == Gather::WIDE) {
        gather_wide<P, L, F, BF16>(a, tab, slots, pts, x);
    } else if (__all(in_unit_cube<3 * P>(pts))) {
        gather_operands<P, L, F, BF16, false, ND, G>(a, tab, pts, x);
    } else {
        gather_operands<P, L, F, BF16, true, ND, G>(a, tab, pts, x);
    }
#pragma unroll
    for (int s = 0; s < K0 / 16; s++) {
        lo[s] = __builtin_bit_cast(V, make_uint4(x[4 * s], x[4 * s + 1], x[4 * s + 2], x[4 * s + 3]));
        const int h = K0 / 4 + 4 * s;
        hi[s] = __builtin_bit_cast(V, make_uint4(x[h], x[h + 1], x[h + 2], x[h + 3]));
        swap_halves(lo[s], hi[s]);
    }
}

// The 8 output rows of this lane's own segment (column lane%32 of column block g), times inv.
// Rows 0..3 of a column block sit in lane group 0, rows 4..7 in lane group 1 (registers 0..3).
__device__ __forceinline__ void gather_logits(const floatx16 out[2], uint32_t g, float inv, float z[8])
{
    float send[4], recv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        send[r] = g ? out[0][r] : out[1][r];
        recv[r] = __shfl_xor(send[r], 32);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        z[r]     = (g ? recv[r] : out[0][r]) * inv;
        z[4 + r] = (g ? out[1][r] : recv[r]) * inv;
    }
}

// ReLU + conversion of the accumulators acc[rb][cb] into the B operands of the next layer.
template <bool BF16>
__device__ __forceinline__ void acc_to_b(const floatx16 acc[2][2], typename Frag<BF16>::vec bh[2][4])
{
    typedef typename Frag<BF16>::elem E;
#pragma unroll
    for (int cb = 0; cb < 2; cb++)
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v = acc[s / 2][cb][8 * (s % 2) + e];
                bh[cb][s][e] = (E)(v > 0.f ? v : 0.f);
            }
}

// The whole network for the 64 segments of a wave. own[3P]: this lane's segment points.
// Returns this lane's 8 logits (descaled). wfrag: LDS fragments (16 B per lane each).
template <int P, int L, int F, bool BF16, int ND, Gather G>
__device__ __forceinline__ void mfma_network(const NetArgs& a, const uint4* __restrict__ wfrag, uint32_t slots,
                                             const float* own, float z[8])
{
    constexpr int K0 = P * L * F;
    typedef MlpShape<K0> S;
    typedef Frag<BF16> FR;
    typedef typename FR::vec V;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t g    = lane >> 5;
    V b1[2][S::KS1];
    layer1_operands<P, L, F, BF16, ND, G>(a, slots, own, b1[0], b1[1]);
    floatx16 acc[2][2];
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int cb = 0; cb < 2; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[rb][cb][r] = 0.f;
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int s = 0; s < S::KS1; s++) {
            const V w = __builtin_bit_cast(V, wfrag[(rb * S::KS1 + s) * 64 + lane]);
            acc[rb][0] = FR::mfma(w, b1[0][s], acc[rb][0]);
            acc[rb][1] = FR::mfma(w, b1[1][s], acc[rb][1]);
        }
    int fbase = S::F_L1;
#pragma unroll
    for (int layer = 0; layer < 3; layer++) {
        V bh[2][4];
        acc_to_b<BF16>(acc, bh);
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int cb = 0; cb < 2; cb++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[rb][cb][r] = 0.f;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const V w = __builtin_bit_cast(V, wfrag[(fbase + rb * 4 + s) * 64 + lane]);
                acc[rb][0] = FR::mfma(w, bh[0][s], acc[rb][0]);
                acc[rb][1] = FR::mfma(w, bh[1][s], acc[rb][1]);
            }
        fbase += S::F_HID;
    }
    floatx16 out[2];
    {
        V bh[2][4];
        acc_to_b<BF16>(acc, bh);
#pragma unroll
        for (int cb = 0; cb < 2; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) out[cb][r] = 0.f;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const V w = __builtin_bit_cast(V, wfrag[(fbase + s) * 64 + lane]);
            out[0] = FR::mfma(w, bh[0][s], out[0]);
            out[1] = FR::mfma(w, bh[1][s], out[1]);
        }
    }
    gather_logits(out, g, a.inv_table_scale, z);
}

// Waves per workgroup of the query kernel; the workgroup shares one LDS copy of the weights.
#ifndef NBVH_MFMA_BLOCK_WAVES
#define NBVH_MFMA_BLOCK_WAVES 4
#endif
constexpr int kWavesPerBlock = NBVH_MFMA_BLOCK_WAVES;

// N elements from global memory into LDS by the whole workgroup: a fixed trip count, so that all
// of a thread's loads are in flight before the first store.
template <int N, typename T>
__device__ __forceinline__ void stage(const T* __restrict__ src, T* lds)
{
    constexpr int B = 64 * kWavesPerBlock;
    constexpr int FULL = N / B;
    const int t = (int)threadIdx.x;
    T v[FULL > 0 ? FULL : 1];
#pragma unroll
    for (int i = 0; i < FULL; i++) v[i] = src[i * B + t];
#pragma unroll
    for (int i = 0; i < FULL; i++) lds[i * B + t] = v[i];
    if (N % B != 0 && FULL * B + t < N) lds[FULL * B + t] = src[FULL * B + t];
}

template <int P, int L, int F, bool BF16>
__device__ __forceinline__ void stage_weights(const NetArgs& a, uint4* wfrag)
{
    constexpr int NF = MlpShape<P * L * F>::N_FRAG;
    const uint4* src = reinterpret_cast<const uint4*>(a.mlp_frag) + (BF16 ? (size_t)NF * 64 : 0);
    stage<NF * 64>(src, wfrag);
    __syncthreads();
}

// ---------------------------------------------------------------------------------------------
// FP8 variant: FP16 first and output layers, e4m3 hidden layers (v_mfma_f32_32x32x16_fp8_fp8).
// Weights of hidden layer l carry a per-layer power-of-two scale (host, amax -> [224, 448)).
// Activations entering an e4m3 layer are scaled per segment (per MFMA column) by a power of two
// that brings the segment's largest activation into [224, 448): the scale depends on the segment
// alone, so results do not depend on what else the wave evaluates. The bias-free ReLU MLP is
// positively homogeneous, so every scale is undone exactly on the logits.
// ---------------------------------------------------------------------------------------------
typedef long fp8x8_t;  // one K = 16 operand per lane: 8 e4m3 values, element e in byte e

struct Fp8Weights {
    static constexpr int kHidden = 3;       // hidden 64x64 layers in e4m3
    static constexpr int kFragsPerLayer = 8;
};

// 2^k with amax * 2^k in [224, 448); 1 for zero, subnormal or non-finite amax.
__device__ __forceinline__ float fp8_column_scale(float amax)
{
    const uint32_t b = __float_as_uint(amax);
    const int e = (int)(b >> 23) - 127;  // amax >= 0 (post-ReLU maximum)
    if (!(amax > 0.f) || e == -127 || e == 128) return 1.f;
    int k = ((b & 0x7FFFFFu) < 0x600000u ? 8 : 7) - e;  // mantissa < 1.75: 2^8 side, else 2^7
    k = k < -126 ? -126 : (k > 127 ? 127 : k);
    return __uint_as_float((uint32_t)(k + 127) << 23);
}

// Per column block: the largest (post-ReLU) activation of this lane's column, over both lane halves.
__device__ __forceinline__ void column_scales(const floatx16 acc[2][2], float sx[2])
{
#pragma unroll
    for (int cb = 0; cb < 2; cb++) {
        float m = 0.f;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) m = fmaxf(m, acc[rb][cb][r]);
        m = fmaxf(m, __shfl_xor(m, 32));
        sx[cb] = fp8_column_scale(m);
    }
}

__device__ __forceinline__ fp8x8_t pack_fp8(const float v[8])
{
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], lo, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], hi, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], hi, true);
    return (fp8x8_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// LDS images of the FP8-variant weights: FP16 layer-1 and output fragments, e4m3 hidden ones.
template <int K0>
struct Fp8Lds {
    uint4 l1[MlpShape<K0>::F_L1 * 64];
    uint4 out[4 * 64];
    uint2 hid[Fp8Weights::kHidden * Fp8Weights::kFragsPerLayer * 64];
};

template <int K0>
__device__ __forceinline__ void stage_weights_fp8(const NetArgs& a, Fp8Lds<K0>& w)
{
    typedef MlpShape<K0> S;
    const uint4* f16 = reinterpret_cast<const uint4*>(a.mlp_frag);
    const uint2* f8  = reinterpret_cast<const uint2*>(a.mlp_frag_fp8);
    stage<S::F_L1 * 64>(f16, w.l1);
    stage<4 * 64>(f16 + (size_t)(S::F_L1 + 3 * S::F_HID) * 64, w.out);
    stage<Fp8Weights::kHidden * Fp8Weights::kFragsPerLayer * 64>(f8, w.hid);
    __syncthreads();
}

template <int P, int L, int F, int ND, Gather G>
__device__ __forceinline__ void mfma_network_fp8(const NetArgs& a, const Fp8Lds<P * L * F>& w, uint32_t slots,
                                                 const float* own, float z[8])
{
    constexpr int K0 = P * L * F;
    typedef MlpShape<K0> S;
    typedef Frag<false> FR;
    typedef typename FR::vec V;
    typedef typename FR::elem E;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t g    = lane >> 5;
    V b1[2][S::KS1];
    layer1_operands<P, L, F, false, ND, G>(a, slots, own, b1[0], b1[1]);
    floatx16 acc[2][2];
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int cb = 0; cb < 2; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[rb][cb][r] = 0.f;
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int s = 0; s < S::KS1; s++) {
            const V wv = __builtin_bit_cast(V, w.l1[(rb * S::KS1 + s) * 64 + lane]);
            acc[rb][0] = FR::mfma(wv, b1[0][s], acc[rb][0]);
            acc[rb][1] = FR::mfma(wv, b1[1][s], acc[rb][1]);
        }
    float cum[2] = {a.table_scale, a.table_scale};  // product of every scale applied, per column block
#pragma unroll
    for (int layer = 0; layer < Fp8Weights::kHidden; layer++) {
        float sx[2];
        column_scales(acc, sx);
        fp8x8_t bh[2][4];
#pragma unroll
        for (int cb = 0; cb < 2; cb++) {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = fmaxf(acc[s / 2][cb][8 * (s % 2) + e], 0.f) * sx[cb];
                bh[cb][s] = pack_fp8(v);
            }
            cum[cb] *= sx[cb] * a.fp8_wscale[layer];
        }
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int cb = 0; cb < 2; cb++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[rb][cb][r] = 0.f;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const fp8x8_t wv = __builtin_bit_cast(
                    fp8x8_t, w.hid[(layer * Fp8Weights::kFragsPerLayer + rb * 4 + s) * 64 + lane]);
                acc[rb][0] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(wv, bh[0][s], acc[rb][0], 0, 0, 0);
                acc[rb][1] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(wv, bh[1][s], acc[rb][1], 0, 0, 0);
            }
    }
    floatx16 out[2];
    {
        float sx[2];
        column_scales(acc, sx);
        V bh[2][4];
#pragma unroll
        for (int cb = 0; cb < 2; cb++) {
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int e = 0; e < 8; e++) bh[cb][s][e] = (E)(fmaxf(acc[s / 2][cb][8 * (s % 2) + e], 0.f) * sx[cb]);
            cum[cb] *= sx[cb];
        }
#pragma unroll
        for (int cb = 0; cb < 2; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) out[cb][r] = 0.f;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const V wv = __builtin_bit_cast(V, w.out[s * 64 + lane]);
            out[0] = FR::mfma(wv, bh[0][s], out[0]);
            out[1] = FR::mfma(wv, bh[1][s], out[1]);
        }
    }
    // cum is a product of powers of two: its reciprocal is exact.
    gather_logits(out, g, 1.f / cum[g], z);
}

// Minimum waves per SIMD the register allocation must allow (latency hiding of the gathers).
#ifndef NBVH_MFMA_WAVES_PER_EU
#define NBVH_MFMA_WAVES_PER_EU 2
#endif

template <int P, int L, int F, bool BF16, bool PARTS, int ND, Gather G>
__global__ __launch_bounds__(64 * kWavesPerBlock, NBVH_MFMA_WAVES_PER_EU) void neural_query_mfma_kernel(NetArgs a,
                                                                                RayBatch b,
                                                                                uint32_t* __restrict__ queue)
{
    constexpr int NF = MlpShape<P * L * F>::N_FRAG;
    __shared__ uint4 wfrag[NF * 64];
    __shared__ uint32_t stack_lds[kWavesPerBlock * kNeuralStackSize * 64];
    __shared__ uint4 node_lds[2 * kNodeCache];
    const uint32_t n_cached = stage_nodes(a, node_lds);
    stage_weights<P, L, F, BF16>(a, wfrag);  // ends with the barrier
    const CachedNodes nodes{a.nodes, node_lds, n_cached};
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    LdsStack st{stack_lds + wave * kNeuralStackSize * 64 + lane, 0};
    RayQueue q;
    q.init(queue, batch_count(b), a.image_width, a.queue_bands);
    Slot s;
    const uint32_t slots = first_rays<PARTS>(a, b, q, s);
    while (fill_slots<PARTS>(a, nodes, s, st, b, q)) {
        float own[3 * P];
        if (s.state == SLOT_SEG) {
            encode_segment(a, s.ray, s.seg_mint, s.seg_maxt, own, &s.rng);
        } else {
#pragma unroll
            for (int c = 0; c < 3 * P; c++) own[c] = 0.5f;
        }
        float z[8];
        mfma_network<P, L, F, BF16, ND, G>(a, wfrag, slots, own, z);
        if (s.state == SLOT_SEG) consume_segment<PARTS>(a, s, z, b);
    }
}

template <int P, int L, int F, bool BF16, int ND>
__global__ __launch_bounds__(64 * kWavesPerBlock, NBVH_MFMA_WAVES_PER_EU) void network_mfma_kernel(NetArgs a, const float* __restrict__ in,
                                                                           uint32_t n, uint32_t group,
                                                                           float* __restrict__ out,
                                                                           float* __restrict__ logits)
{
    constexpr int NF = MlpShape<P * L * F>::N_FRAG;
    __shared__ uint4 wfrag[NF * 64];
    stage_weights<P, L, F, BF16>(a, wfrag);
    // Persistent over chunks of `group` inputs, a multiple of 64 up to blockDim.x (network_waves), so
    // that every lane of a working wave takes part in each MFMA; the weights are staged once per
    // resident workgroup, by all its waves.
    if (threadIdx.x >= group) return;
    for (uint32_t base = blockIdx.x * group; base < n; base = next_chunk(base, group, n)) {
        asm volatile("" ::: "memory");  // keeps the weights' LDS reads in the loop (hoisted: one wave per SIMD)
        const uint32_t i = base + threadIdx.x;
        float own[3 * P];
#pragma unroll
        for (int c = 0; c < 3 * P; c++) own[c] = i < n ? in[(size_t)i * (3 * P) + c] : 0.5f;
        float z[8];
        mfma_network<P, L, F, BF16, ND, kNetworkGather<L, ND>>(a, wfrag, 64u, own, z);
        if (i < n) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (out) out[(size_t)i * 8 + j] = sigmoidf_cw(z[j]);
                if (logits) logits[(size_t)i * 8 + j] = z[j];
            }
        }
    }
}

template <int P, int L, int F, bool PARTS, int ND, Gather G>
__global__ __launch_bounds__(64 * kWavesPerBlock, NBVH_MFMA_WAVES_PER_EU) void neural_query_fp8_kernel(NetArgs a,
                                                                               RayBatch b,
                                                                               uint32_t* __restrict__ queue)
{
    __shared__ Fp8Lds<P * L * F> w;
    __shared__ uint32_t stack_lds[kWavesPerBlock * kNeuralStackSize * 64];
    __shared__ uint4 node_lds[2 * kNodeCache];
    const uint32_t n_cached = stage_nodes(a, node_lds);
    stage_weights_fp8<P * L * F>(a, w);  // ends with the barrier
    const CachedNodes nodes{a.nodes, node_lds, n_cached};
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    LdsStack st{stack_lds + wave * kNeuralStackSize * 64 + lane, 0};
    RayQueue q;
    q.init(queue, batch_count(b), a.image_width, a.queue_bands);
    Slot s;
    const uint32_t slots = first_rays<PARTS>(a, b, q, s);
    while (fill_slots<PARTS>(a, nodes, s, st, b, q)) {
        float own[3 * P];
        if (s.state == SLOT_SEG) {
            encode_segment(a, s.ray, s.seg_mint, s.seg_maxt, own, &s.rng);
        } else {
#pragma unroll
            for (int c = 0; c < 3 * P; c++) own[c] = 0.5f;
        }
        float z[8];
        mfma_network_fp8<P, L, F, ND, G>(a, w, slots, own, z);
        if (s.state == SLOT_SEG) consume_segment<PARTS>(a, s, z, b);
    }
}

template <int P, int L, int F, int ND>
__global__ __launch_bounds__(64 * kWavesPerBlock, NBVH_MFMA_WAVES_PER_EU) void network_fp8_kernel(NetArgs a, const float* __restrict__ in,
                                                                          uint32_t n, uint32_t group,
                                                                          float* __restrict__ out,
                                                                          float* __restrict__ logits)
{
    __shared__ Fp8Lds<P * L * F> w;
    stage_weights_fp8<P * L * F>(a, w);
    if (threadIdx.x >= group) return;
    for (uint32_t base = blockIdx.x * group; base < n; base = next_chunk(base, group, n)) {
        asm volatile("" ::: "memory");  // keeps the weights' LDS reads in the loop (hoisted: one wave per SIMD)
        const uint32_t i = base + threadIdx.x;
        float own[3 * P];
#pragma unroll
        for (int c = 0; c < 3 * P; c++) own[c] = i < n ? in[(size_t)i * (3 * P) + c] : 0.5f;
        float z[8];
        mfma_network_fp8<P, L, F, ND, kNetworkGather<L, ND>>(a, w, 64u, own, z);
        if (i < n) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (out) out[(size_t)i * 8 + j] = sigmoidf_cw(z[j]);
                if (logits) logits[(size_t)i * 8 + j] = z[j];
            }
        }
    }
}

}  // namespace dev

namespace {

// PREC: NBVH_PREC_FP16, _BF16 or _FP8.
template <int P, int L, int F, uint32_t PREC, bool PARTS, int ND, dev::Gather G>
auto query_kernel()
{
    if constexpr (PREC == NBVH_PREC_FP8)
        return dev::neural_query_fp8_kernel<P, L, F, PARTS, ND, G>;
    else
        return dev::neural_query_mfma_kernel<P, L, F, PREC == NBVH_PREC_BF16, PARTS, ND, G>;
}

template <int P, int L, int F, uint32_t PREC, bool PARTS>
hipError_t launch_query_k(const NetArgs& a, const RayBatch& rb, uint32_t* queue, uint32_t n_cus, hipStream_t stream,
                          QueryGrid* plan)
{
    using dev::Gather;
    constexpr uint32_t threads = 64 * dev::kWavesPerBlock;
    constexpr int ND = kDensePrefix;
    const auto wide  = query_kernel<P, L, F, PREC, PARTS, -1, Gather::WIDE>();
    const auto dense = query_kernel<P, L, F, PREC, PARTS, ND, dev::kQueryGather<L, ND>>();
    const auto any   = query_kernel<P, L, F, PREC, PARTS, -1, Gather::LEVELS>();
    // Every variant is bounded to two waves per SIMD and holds the same LDS.
    static const uint32_t bpc = blocks_per_cu(any, threads);
    const uint32_t cap = a.blocks_per_cu != 0u && a.blocks_per_cu < bpc ? a.blocks_per_cu : bpc;
    const QueryGrid g = query_grid(rb, dev::kWavesPerBlock, n_cus * cap, 64u / L, 16u);
    if (plan) {
        *plan = g;
        return hipSuccess;
    }
    NetArgs args = a;
    args.static_slots = g.static_slots;
    if (g.static_slots == 0u) {
        const hipError_t e = zero_u32(queue, dev::kQueueWords, stream);
        if (e != hipSuccess) return e;
    }
    // Static launches have few waves per CU and want loads in flight, not a common level: 48,240
    // rays 264 us before level order, 246 us by pairs; 65,536 rays 270 us by phases, 259 by levels.
    // 8 x 4 grid by pairs: 65,536 rays 168 -> 137 us, 131,072 214 -> 166. General grids by pairs: 374
    // against 381 us (16 x 2 with 2^21 entries, 100,000 rays), others up to 3 % slower; left as they were.
    const auto few = query_kernel<P, L, F, PREC, PARTS, ND, Gather::PAIRS>();
    const auto k = g.wide ? wide : a.n_dense == (uint32_t)ND ? (g.static_slots ? few : dense) : any;
    hipLaunchKernelGGL(k, dim3(g.blocks), dim3(threads), 0, stream, args, rb, queue);
    return hipGetLastError();
}

template <int P, int L, int F, uint32_t PREC>
hipError_t launch_query(const NetArgs& a, const RayBatch& rb, uint32_t* queue, uint32_t n_cus, hipStream_t stream,
                        QueryGrid* plan)
{
    return rb.parts ? launch_query_k<P, L, F, PREC, true>(a, rb, queue, n_cus, stream, plan)
                    : launch_query_k<P, L, F, PREC, false>(a, rb, queue, n_cus, stream, plan);
}

template <int P, int L, int F, bool BF16, int ND>
hipError_t launch_network_nd(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits, uint32_t n_cus,
                             hipStream_t stream)
{
    auto k = dev::network_mfma_kernel<P, L, F, BF16, ND>;
    static const uint32_t bpc = blocks_per_cu(k, 64 * dev::kWavesPerBlock);
    const uint32_t resident = n_cus * bpc, group = 64u * network_waves(n, dev::kWavesPerBlock, resident);
    uint32_t blocks = n / group + (n % group != 0u ? 1u : 0u);
    blocks = blocks < resident ? blocks : resident;
    hipLaunchKernelGGL(k, dim3(blocks), dim3(64 * dev::kWavesPerBlock), 0, stream, a, in, n, group, out, logits);
    return hipGetLastError();
}

template <int P, int L, int F, bool BF16>
hipError_t launch_network(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits, uint32_t n_cus,
                          hipStream_t stream)
{
    return a.n_dense == (uint32_t)kDensePrefix
               ? launch_network_nd<P, L, F, BF16, kDensePrefix>(a, in, n, out, logits, n_cus, stream)
               : launch_network_nd<P, L, F, BF16, -1>(a, in, n, out, logits, n_cus, stream);
}

template <int P, int L, int F, int ND>
hipError_t launch_network_fp8_nd(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits,
                                 uint32_t n_cus, hipStream_t stream)
{
    auto k = dev::network_fp8_kernel<P, L, F, ND>;
    static const uint32_t bpc = blocks_per_cu(k, 64 * dev::kWavesPerBlock);
    const uint32_t resident = n_cus * bpc, group = 64u * network_waves(n, dev::kWavesPerBlock, resident);
    uint32_t blocks = n / group + (n % group != 0u ? 1u : 0u);
    blocks = blocks < resident ? blocks : resident;
    hipLaunchKernelGGL(k, dim3(blocks), dim3(64 * dev::kWavesPerBlock), 0, stream, a, in, n, group, out, logits);
    return hipGetLastError();
}

template <int P, int L, int F>
hipError_t launch_network_fp8(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits, uint32_t n_cus,
                              hipStream_t stream)
{
    return a.n_dense == (uint32_t)kDensePrefix
               ? launch_network_fp8_nd<P, L, F, kDensePrefix>(a, in, n, out, logits, n_cus, stream)
               : launch_network_fp8_nd<P, L, F, -1>(a, in, n, out, logits, n_cus, stream);
}

}  // namespace

#define NBVH_MFMA_SHAPES(X) X(3, 16, 2) X(3, 8, 4)

hipError_t query_mfma(const NetArgs& a, uint32_t precision, const RayBatch& rb, uint32_t* queue, uint32_t n_cus,
                      hipStream_t stream, bool* supported, QueryGrid* plan)
{
    *supported = true;
    if (a.n_hidden_layers == 4 && a.mlp_frag != nullptr && a.tables_f16_bytes != 0) {
#define X(P_, L_, F_)                                                                       \
    if (a.n_points == P_ && a.n_levels == L_ && a.n_features == F_) {                      \
        if (precision == NBVH_PREC_FP16)                                                   \
            return launch_query<P_, L_, F_, NBVH_PREC_FP16>(a, rb, queue, n_cus, stream, plan);  \
        if (precision == NBVH_PREC_BF16)                                                   \
            return launch_query<P_, L_, F_, NBVH_PREC_BF16>(a, rb, queue, n_cus, stream, plan);  \
        if (precision == NBVH_PREC_FP8 && a.mlp_frag_fp8 != nullptr)                       \
            return launch_query<P_, L_, F_, NBVH_PREC_FP8>(a, rb, queue, n_cus, stream, plan);   \
    }
        NBVH_MFMA_SHAPES(X)
#undef X
    }
    *supported = false;
    return hipSuccess;
}

hipError_t network_mfma(const NetArgs& a, uint32_t precision, const float* in, uint32_t n, float* out, float* logits,
                        uint32_t n_cus, hipStream_t stream, bool* supported)
{
    *supported = true;
    if (a.n_hidden_layers == 4 && a.mlp_frag != nullptr && a.tables_f16_bytes != 0) {
#define X(P_, L_, F_)                                                                 \
    if (a.n_points == P_ && a.n_levels == L_ && a.n_features == F_) {                \
        if (precision == NBVH_PREC_FP16)                                             \
            return launch_network<P_, L_, F_, false>(a, in, n, out, logits, n_cus, stream);  \
        if (precision == NBVH_PREC_BF16)                                             \
            return launch_network<P_, L_, F_, true>(a, in, n, out, logits, n_cus, stream);   \
        if (precision == NBVH_PREC_FP8 && a.mlp_frag_fp8 != nullptr)                 \
            return launch_network_fp8<P_, L_, F_>(a, in, n, out, logits, n_cus, stream);     \
    }
        NBVH_MFMA_SHAPES(X)
#undef X
    }
    *supported = false;
    return hipSuccess;
}

}  // namespace nbvh
