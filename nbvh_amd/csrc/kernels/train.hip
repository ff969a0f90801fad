// train.hip -- one training step of the network on encoded segments and their targets: the
// replacement of the reference's trainer->training_step(stream, inputs[9 x n], targets[8 x n])
// (src/cuda/neural/neural_bvh_renderer.cu:170-173) for its default configuration. FP32 throughout.
//
// Workspace: 720 activation rows of act_stride floats each (row r, sample i at r * stride + i),
// the weight fragments of the two passes, and per-chunk partial matrix gradients.
//   train_fragments  the matrices as MFMA operands of the forward and the backward pass;
//   train_forward    32 samples per wave: hash-grid features (two lanes per sample share the
//                    levels) and the MLP on the FP32 matrix cores; every layer's outputs go to the
//                    activation rows;
//   train_backward   the composite loss of the reference's defaults (pt_composite_loss.cuh:19-123,
//                    neural_bvh_module.h:250-266), its gradient through the Sigmoid outputs and the
//                    ReLU layers (transposed fragments), stored per layer, down to the feature
//                    gradients;
//   train_scatter    the table gradient of levels of fewer than 128 slices of 128 KB, one
//                    workgroup per slice: the slice is summed in LDS from every (sample, point)
//                    whose corners fall in it and stored whole;
//   train_bin_*      the table gradient of the other levels: the corner terms binned by slice
//                    (count, scan, scatter), then one workgroup per slice sums its bin in LDS
//                    and stores the slice whole; no global atomics on the gradient;
//   train_wgrad      the matrix gradients dW[o][i] = sum over samples of delta[o] * act[i]: each
//                    workgroup reduces one chunk of samples for one matrix on the matrix cores
//                    through LDS tiles of 32 samples and writes its partial; train_wgrad_reduce adds the partials in
//                    chunk order (deterministic);
//   train_adam       tiny-cuda-nn's Adam: per-parameter update counts for the bias correction,
//                    L2 regularisation and dense updates for the matrices, sparse updates
//                    without L2 for the tables (entries no sample touched keep their value).
// Gradients are sums over the batch of the per-element gradients divided by n * 8, as the
// reference's loss kernel writes them; the table gradients are summed by atomics in an order that
// is not fixed, everything else in a fixed one. Training amplifies that order: four steps of 10,007
// samples on the 8 x 4 grid, repeated from the same state, give the same first step but for the
// table gradient's last bits, and then matrices that differ by 2e-8 to 6e-4 (by seed; a ReLU or an
// L1 sign decided the other way), and losses by up to 4e-6.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../device/mlp_f32.h"
#include "launch.h"

namespace nbvh {
namespace dev {

constexpr int kK0 = 96, kH = 64, kO = 8, kLayers = 5;
// Activation rows: a0 (features) | h1..h4 | y | d1..d4 (deltas of h1..h4) | d5 (delta of y) |
// dx (feature gradients).
constexpr int kA0 = 0, kHid = kA0 + kK0, kY = kHid + 4 * kH, kD = kY + kO, kD5 = kD + 4 * kH, kDX = kD5 + kO;
constexpr int kRows   = kDX + kK0;                          // 720 rows
#ifndef NBVH_SCATTER_SLICE_FLOATS
#define NBVH_SCATTER_SLICE_FLOATS 32768
#endif
constexpr int kSliceFloats = NBVH_SCATTER_SLICE_FLOATS;     // table-gradient slice in LDS (128 KB)
constexpr uint32_t kScatterThreads = 1024;                  // threads sharing one slice
#ifndef NBVH_SCATTER_UNROLL
#define NBVH_SCATTER_UNROLL 2                               // (sample, point) pairs per thread and iteration
#endif
constexpr int kMlp    = kH * kK0 + 3 * kH * kH + kO * kH;  // 18,944 matrix entries
constexpr int kChunks = 256;                                // most matrix-gradient partials

__host__ __device__ constexpr int w_offset(int layer)
{
    return layer == 0 ? 0 : kH * kK0 + (layer - 1) * kH * kH;
}

__device__ __forceinline__ float& row(float* act, size_t stride, int r, uint32_t i)
{
    return act[(size_t)r * stride + i];
}

// MLP weight fragments of a step: the forward ones in the layout of device/mlp_f32.h
// (F32Layout<96>), then the backward ones: matrix l transposed, rows = its inputs, k-steps over
// its outputs. Per matrix: row block, pair of k-steps, lane, k-step of the pair, as in the forward
// layout; inputs are ordered within a block of 32 rows like the forward rows (row 8 q + 4 g + i is
// input 2 (16 rb + 4 q + i) + g), so that accumulators are the next product's B operands here too.
__host__ __device__ constexpr int wt_offset(int layer)  // matrix 4 first: the order of the backward pass
{
    return layer == 4 ? 0 : layer == 3 ? kH * kO : kH * kO + (3 - layer) * kH * kH;
}

__global__ __launch_bounds__(256) void train_fragments_kernel(const float* __restrict__ mlp, float* __restrict__ wf,
                                                              float* __restrict__ wb)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= kMlp) return;
    const int layer = j < w_offset(1) ? 0 : j < w_offset(4) ? 1 + (j - w_offset(1)) / (kH * kH) : 4;
    const int out_w = layer == 4 ? kO : kH, in_w = layer == 0 ? kK0 : kH;
    const int local = j - w_offset(layer), o = local / in_w, k = local % in_w;
    const float w = mlp[j];
    // Row of neuron (or input) n in its block of 32, and the block.
    auto row_of = [](int n, int& rb) {
        const int g = n & 1, m = n >> 1;
        rb = m / 16;
        return 8 * ((m % 16) / 4) + 4 * g + m % 4;
    };
    auto at = [](int steps, int rb, int row, int kk) {
        const int s = kk >> 1, g = kk & 1;
        return ((rb * (steps / 2) + s / 2) * 64 + g * 32 + row) * 2 + (s & 1);
    };
    int rb;
    if (layer < 4) {
        const int row = row_of(o, rb);
        wf[w_offset(layer) + at(in_w / 2, rb, row, k)] = w;
    } else {
        const int st = k >> 1, g = k & 1;
        wf[w_offset(4) + ((st / 2 * 2 + g) * 8 + o) * 2 + (st & 1)] = w;
    }
    const int row = row_of(k, rb);
    wb[wt_offset(layer) + at(out_w / 2, rb, row, o)] = w;
}

// A wave takes 32 samples (one MFMA block of segments): both lanes l and l + 32 work for sample
// l, so 65,536 samples are two waves per SIMD of the whole chip. Workgroups of 8 waves (256
// samples) share one LDS copy of the weight fragments; small batches take 2-wave workgroups so
// that they reach every CU.
constexpr int kWaveSamples = 32;
constexpr uint32_t kSmallBatch = 32768;
constexpr uint32_t kMinGroup   = 2 * kWaveSamples;  // samples of the smaller workgroup

// Features of sample l on lanes l (even levels) and l + 32 (odd levels), as the B operands of layer
// 1: x[s] holds feature 2 s on lanes 0..31 and 2 s + 1 on lanes 32..63 (one v_permlane32_swap per
// two k-steps). Every sum runs over corners 0..7 in order.
template <int P, int L, int F, bool EXACT>
__device__ __forceinline__ void half_features(const NetArgs& a, const float* __restrict__ tables, const float* pts,
                                              float* x)
{
    const uint32_t g = (threadIdx.x >> 5) & 1u;
#pragma unroll
    for (int l0 = 0; l0 < L; l0 += 2) {
        const GridLevel &v0 = a.level[l0], &v1 = a.level[l0 + 1];
        const GridLevel lv{g ? v1.scale : v0.scale, g ? v1.res : v0.res,       g ? v1.res2 : v0.res2,
                           g ? v1.size : v0.size,   g ? v1.offset : v0.offset, g ? v1.dense : v0.dense};
        float f[P * F];
        if (!v0.dense && !v1.dense)  // uniform
            gather_level_f32<P, F, true, false>(lv, tables, pts, f);
        else
            gather_level_f32<P, F, false, EXACT>(lv, tables, pts, f);
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int k = 0; k < F; k += 2) {
                const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(f[p * F + k]),
                                                                __float_as_uint(f[p * F + k + 1]), false, false);
                x[(p * L + l0) * (F / 2) + k / 2]     = __uint_as_float(r[0]);
                x[(p * L + l0 + 1) * (F / 2) + k / 2] = __uint_as_float(r[1]);
            }
    }
}

// acc[rb] += (RB blocks of 32 rows of the S k-steps' weights) x b[s].
template <int S, int RB>
__device__ __forceinline__ void train_layer(const float* w, const float* b, floatx16_t* acc)
{
    const float2* w2 = reinterpret_cast<const float2*>(w) + (threadIdx.x & 63u);
#pragma unroll
    for (int s = 0; s < S; s += 2) {
        float2 v[RB];
#pragma unroll
        for (int rb = 0; rb < RB; rb++) v[rb] = w2[(rb * (S / 2) + s / 2) * 64];
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x2f32(e ? v[rb].y : v[rb].x, b[s + e], acc[rb], 0, 0, 0);
    }
}

// The forward pass on the FP32 matrix cores (bit-identical to fmaf chains with k ascending, see
// device/mlp_f32.h). Per layer the 64 activations of a sample sit in two lanes, k = 2 s + l / 32 in
// register s, which are stored to the activation rows (128 B per half wave) and feed the next layer.
// Measured per 65,536 samples of the 16 x 2 grid: 167 us, against 258 us with one thread per
// sample and weights through the scalar cache; what is left is the gathers and 94 MB of rows.
template <int P, int L, int F, int W>
__global__ __launch_bounds__(64 * W, 2) void train_forward_kernel(TrainArgs t, const float* __restrict__ wf,
                                                                 const float* __restrict__ in,
                                                                 float* __restrict__ act, uint32_t n)
{
    __shared__ float4 w_lds[kMlp / 4];
    for (uint32_t j = threadIdx.x; j < (uint32_t)kMlp / 4u; j += 64u * W)
        w_lds[j] = reinterpret_cast<const float4*>(wf)[j];
    const uint32_t lane = threadIdx.x & 63u, g = lane >> 5;
    const uint32_t i = (blockIdx.x * W + (threadIdx.x >> 6)) * kWaveSamples + (lane & 31u);
    const size_t S = t.act_stride;
    const bool ok = i < n;
    float pts[3 * P], x[kK0 / 2];
#pragma unroll
    for (int c = 0; c < 3 * P; c++) pts[c] = ok ? in[(size_t)i * (3 * P) + c] : 0.5f;
    if (__all(in_unit_cube<3 * P>(pts)))
        half_features<P, L, F, false>(t.net, t.tables, pts, x);
    else
        half_features<P, L, F, true>(t.net, t.tables, pts, x);
    __syncthreads();
    const float* w = reinterpret_cast<const float*>(w_lds);
    if (ok) {
#pragma unroll
        for (int s = 0; s < kK0 / 2; s++) row(act, S, kA0 + 2 * s + g, i) = x[s];
    }
    floatx16_t acc[2] = {};
    train_layer<kK0 / 2, 2>(w, x, acc);
    float b[kH / 2];
#pragma unroll
    for (int layer = 0; layer < 4; layer++) {
#pragma unroll
        for (int s = 0; s < kH / 2; s++) b[s] = fmaxf(acc[s / 16][s % 16], 0.f);
        if (ok) {
#pragma unroll
            for (int s = 0; s < kH / 2; s++) row(act, S, kHid + layer * kH + 2 * s + g, i) = b[s];
        }
        if (layer == 3) break;
        acc[0] = acc[1] = floatx16_t{};
        train_layer<kH / 2, 2>(w + w_offset(layer + 1), b, acc);
    }
    floatx16_t out = {};
    const float2* wo = reinterpret_cast<const float2*>(w + w_offset(4));
#pragma unroll
    for (int s = 0; s < kH / 2; s += 2) {
        const float2 v = wo[(s + g) * 8 + (lane & 7u)];
        out = __builtin_amdgcn_mfma_f32_32x32x2f32(v.x, b[s], out, 0, 0, 0);
        out = __builtin_amdgcn_mfma_f32_32x32x2f32(v.y, b[s + 1], out, 0, 0, 0);
    }
    if (ok) {
#pragma unroll
        for (int r = 0; r < 4; r++) row(act, S, kY + 4 * g + r, i) = sigmoidf_cw(out[r]);
    }
}

// Loss and gradient of one output element (the reference's defaults; see oracle/train.py).
__device__ __forceinline__ void element_loss(int j, float y, float target, bool keep, float& loss, float& grad)
{
    loss = 0.f;
    grad = 0.f;
    if (j == 0) {  // BinaryCrossEntropy, prediction clamped to [1e-5, 1 - 1e-5]
        const float p = fminf(fmaxf(y, 1e-5f), 1.f - 1e-5f);
        loss = -(target * logf(p) + (1.f - target) * logf(1.f - p));
        grad = -(target - p) / (p - p * p);
    } else if (!keep) {
        return;  // visibility masking: target visibility < 0.5
    } else if (j == 1) {  // depth: L1
        const float d = y - target;
        loss = fabsf(d);
        grad = copysignf(1.f, d);
    } else if (j < 5) {  // normal: L1 on the linearised output ((y*2-1)/0.1)*0.5+0.5, gradient / 0.1
        const float lin = ((y * 2.f - 1.f) / 0.1f) * 0.5f + 0.5f;
        const float d   = lin - target;
        loss = fabsf(d);
        grad = copysignf(1.f, d) * (1.f / 0.1f);
    } else {  // albedo: relative L2 with the denominator held constant
        const float d   = y - target;
        const float den = y * y + 1e-2f;
        loss = d * d / den;
        grad = 2.f * d / den;
    }
}

// The backward pass, 32 samples per wave like the forward pass: delta of layer l - 1 = W_l^T delta_l
// where the activation is positive, with the outputs o ascending (the transposed fragments).
// Measured per 65,536 samples: 82 us (154 us with one thread per sample); 164 MB of rows.
template <int W>
__global__ __launch_bounds__(64 * W, 2) void train_backward_kernel(TrainArgs t, const float* __restrict__ wb,
                                                                  const float* __restrict__ targets,
                                                                  float* __restrict__ act,
                                                                  double* __restrict__ losses, uint32_t n)
{
    __shared__ float4 w_lds[kMlp / 4];
    __shared__ double l_lds[W];
    for (uint32_t j = threadIdx.x; j < (uint32_t)kMlp / 4u; j += 64u * W)
        w_lds[j] = reinterpret_cast<const float4*>(wb)[j];
    const uint32_t lane = threadIdx.x & 63u, g = lane >> 5;
    const uint32_t i = (blockIdx.x * W + (threadIdx.x >> 6)) * kWaveSamples + (lane & 31u);
    const size_t S = t.act_stride;
    const bool ok = i < n;
    const float inv_n = 1.f / ((float)n * (float)kO);
    // Both lanes of a sample form its 8 output deltas; lane l + 32 keeps the odd ones.
    float dz[kO], lsum = 0.f;
#pragma unroll
    for (int j = 0; j < kO; j++) dz[j] = 0.f;
    if (ok) {
        const bool keep = targets[(size_t)i * kO] >= 0.5f;
#pragma unroll
        for (int j = 0; j < kO; j++) {
            const float y = row(act, S, kY + j, i);
            float l, gr;
            element_loss(j, y, targets[(size_t)i * kO + j], keep, l, gr);
            lsum += l * inv_n;
            dz[j] = (gr * inv_n) * (y * (1.f - y));  // through the Sigmoid output activation
        }
        if (t.sample_loss && g == 0u) t.sample_loss[i] = lsum;  // the element values in element order
    }
    float b[kH / 2];
#pragma unroll
    for (int s = 0; s < kO / 2; s++) b[s] = g ? dz[2 * s + 1] : dz[2 * s];
    if (ok) {
#pragma unroll
        for (int s = 0; s < kO / 2; s++) row(act, S, kD5 + 2 * s + g, i) = b[s];
    }
    // The workgroup's loss in double, waves in order; train_wgrad_reduce adds the workgroups'. One
    // float atomic per wave instead: 102 us, and off by 2 ulp at 65,536 samples.
    double wsum = g == 0u ? (double)lsum : 0.0;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) wsum += __shfl_xor(wsum, off);
    if (lane == 0) l_lds[threadIdx.x >> 6] = wsum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < W; k++) s += l_lds[k];
        losses[blockIdx.x] = s;
    }
    const float* w = reinterpret_cast<const float*>(w_lds);
#pragma unroll
    for (int layer = 3; layer >= 0; layer--) {  // delta of h(layer + 1)
        float h[kH / 2];
#pragma unroll
        for (int s = 0; s < kH / 2; s++) h[s] = ok ? row(act, S, kHid + layer * kH + 2 * s + g, i) : 0.f;
        floatx16_t acc[2] = {};
        if (layer == 3)
            train_layer<kO / 2, 2>(w + wt_offset(4), b, acc);
        else
            train_layer<kH / 2, 2>(w + wt_offset(layer + 1), b, acc);
#pragma unroll
        for (int s = 0; s < kH / 2; s++) b[s] = h[s] > 0.f ? acc[s / 16][s % 16] : 0.f;
        if (ok) {
#pragma unroll
            for (int s = 0; s < kH / 2; s++) row(act, S, kD + layer * kH + 2 * s + g, i) = b[s];
        }
    }
    // Feature gradients; train_scatter adds them into the tables' gradient.
    floatx16_t acc[3] = {};
    train_layer<kH / 2, 3>(w + wt_offset(0), b, acc);
    if (ok) {
#pragma unroll
        for (int s = 0; s < kK0 / 2; s++) row(act, S, kDX + 2 * s + g, i) = acc[s / 16][s % 16];
    }
}

// Work items of the table gradient. Slice j of level l holds the level's entries
// [j * E, min((j + 1) * E, size)), E = kSliceFloats / F; each slice is split into parts[l] parts
// of the batch's (sample, point) pairs; level l's items are [first[l], first[l + 1]), item
// first[l] + j * parts[l] + k being part k of slice j.
struct SliceMap {
    uint32_t first[kMaxLevels + 1];
    uint32_t parts[kMaxLevels];
};

// One workgroup per item: the slice's gradient accumulates in LDS while the workgroup visits its
// part of the batch's (sample, point) pairs, recomputes the cell at the slice's level and adds
// w_c * dx[f] for each corner c whose entry lies in the slice (LDS atomics). A slice of a single
// part is then stored whole, zeros included; the parts of a split slice add their non-zero
// entries to the (zeroed) gradient with global atomics. Every entry of every level belongs to
// exactly one slice, so the table gradient is written completely. The cost is a scan of the
// batch's points per item instead of one global atomic add per (point, level, corner, feature);
// slices of the coarse dense levels, which receive many corners, are split so that no workgroup
// adds many more corners than the others.
template <int P, int L, int F>
__global__ __launch_bounds__(kScatterThreads) void train_scatter_kernel(TrainArgs t, SliceMap map,
                                                                        const float* __restrict__ in,
                                                                        const float* __restrict__ act,
                                                                        float* __restrict__ gtab, uint32_t n)
{
    constexpr uint32_t E = kSliceFloats / F;
    __shared__ float acc[kSliceFloats];
    int l = 0;
    while (l + 1 < L && blockIdx.x >= map.first[l + 1]) l++;
    const GridLevel& lv = t.net.level[l];
    const uint32_t parts = map.parts[l], item = blockIdx.x - map.first[l];
    const uint32_t slice = item / parts, part = item - slice * parts;
    const uint32_t e0 = slice * E;
    const uint32_t len = lv.size - e0 < E ? lv.size - e0 : E;
    for (uint32_t j = threadIdx.x; j < len * F; j += kScatterThreads) acc[j] = 0.f;
    __syncthreads();
    const size_t S = t.act_stride;
    const uint32_t total = n * (uint32_t)P;
    const uint32_t j0 = (uint32_t)((uint64_t)total * part / parts), j1 = (uint32_t)((uint64_t)total * (part + 1) / parts);
    // U (sample, point) pairs per thread and iteration, their point loads issued together.
    constexpr uint32_t B = kScatterThreads;
    constexpr int U = NBVH_SCATTER_UNROLL;
    for (uint32_t j = j0 + threadIdx.x; j < j1; j += U * B) {
        float pts[U][3];
#pragma unroll
        for (int h = 0; h < U; h++) {
            const uint32_t jj = j + h * B < j1 ? j + h * B : j;
            const uint32_t i = jj / P, p = jj - i * P;
#pragma unroll
            for (int c = 0; c < 3; c++) pts[h][c] = in[(size_t)i * (3 * P) + 3 * p + c];
        }
#pragma unroll
        for (int h = 0; h < U; h++) {
            const uint32_t jj = j + h * B;
            if (jj >= j1) break;
            const uint32_t i = jj / P, p = jj - i * P;
            uint32_t g[3], idx[8];
            float fr[3];
            grid_cell(lv, pts[h][0], pts[h][1], pts[h][2], g, fr);
            if (!lv.dense)  // uniform per workgroup: only the level's own index formula
                hash_corners(lv, g, idx);
            else if (in_unit_cube<3>(pts[h]))
                grid_corners<false>(lv, g, idx);
            else
                grid_corners<true>(lv, g, idx);
            bool any = false;
#pragma unroll
            for (int c = 0; c < 8; c++) any = any || (idx[c] - e0 < len);
            if (!any) continue;
            float dx[F];
#pragma unroll
            for (int f = 0; f < F; f++) dx[f] = act[(size_t)(kDX + (p * L + l) * F + f) * S + i];
#pragma unroll
            for (uint32_t c = 0; c < 8; c++) {
                const uint32_t r = idx[c] - e0;
                if (r < len) {
                    const float w = corner_weight(c, fr);
#pragma unroll
                    for (int f = 0; f < F; f++) atomicAdd(&acc[r * F + f], w * dx[f]);
                }
            }
        }
    }
    __syncthreads();
    float* out = gtab + ((size_t)lv.offset + e0) * F;
    if (parts == 1) {
        for (uint32_t j = threadIdx.x; j < len * F; j += B) out[j] = acc[j];
    } else {
        for (uint32_t j = threadIdx.x; j < len * F; j += B)
            if (acc[j] != 0.f) atomicAdd(out + j, acc[j]);
    }
}

// Binned table gradient, for levels of 128 or more 128 KB slices: the level is cut into bins of
// kBinFloats gradient floats; every corner term (entry, w_c * dx[f]) of the level is written to
// its bin, then one workgroup per bin adds the bin's terms in LDS and stores the bin whole. Four
// passes:
//   train_bin_count_kernel    per workgroup a histogram of its pairs' corner bins in LDS, added to
//                             the bin counts (one global atomic per workgroup and bin touched);
//   train_bin_scan_kernel     exclusive scan of the counts: bin b's terms at [offsets[b],
//                             offsets[b + 1]); the cursors start at the offsets;
//   train_bin_scatter_kernel  the same pairs again: each workgroup reserves its range of every
//                             bin (one global atomic per bin touched) and writes its terms;
//   train_bin_accumulate_kernel  one workgroup per bin: LDS sum, the bin stored whole.
// The batch is read three times and each term twice, instead of one global atomic add per
// (pair, corner, feature) or one scan of the batch per slice.
struct BinMap {
    uint32_t count;                    // binned levels
    uint32_t level[kMaxLevels];        // their indices
    uint32_t first[kMaxLevels + 1];    // first bin of binned level k; first[count] = bins
};
#ifndef NBVH_BIN_THREADS
#define NBVH_BIN_THREADS 256
#endif
// 8192 pairs: a workgroup's terms reach each bin in runs long enough to write coalesced. Measured
// per step at 2^21 / 2^22 / 2^23 entries (256 threads): 2048 pairs 1.74 / 2.14 / 2.68 ms, 8192
// pairs 1.61 / 2.02 / 2.56 ms (1024 threads: 1.59 / 2.07 / 2.62).
#ifndef NBVH_BIN_PAIRS
#define NBVH_BIN_PAIRS 8192
#endif
constexpr uint32_t kBinThreads = NBVH_BIN_THREADS;
constexpr uint32_t kBinPairs   = NBVH_BIN_PAIRS;  // (sample, point) pairs per workgroup and level
constexpr uint32_t kBinFloats  = 16384;   // gradient floats per bin (64 KB of LDS: 2 workgroups per CU)
constexpr uint32_t kBinWindow  = 8192;    // bins of one level a count / scatter workgroup handles
constexpr uint32_t kBinUnroll  = 4;       // terms per thread whose loads are issued together

// Corners and fractional position of pair jj = (sample i, point p) at level lv.
template <int P>
__device__ __forceinline__ void pair_corners(const GridLevel& lv, const float* __restrict__ in, uint32_t i, uint32_t p,
                                             uint32_t idx[8], float fr[3])
{
    float pt[3];
#pragma unroll
    for (int c = 0; c < 3; c++) pt[c] = in[(size_t)i * (3 * P) + 3 * p + c];
    uint32_t g[3];
    grid_cell(lv, pt[0], pt[1], pt[2], g, fr);
    if (!lv.dense)
        hash_corners(lv, g, idx);
    else if (in_unit_cube<3>(pt))
        grid_corners<false>(lv, g, idx);
    else
        grid_corners<true>(lv, g, idx);
}

// Workgroup (x, k, w): pairs [x * kBinPairs, ...) of binned level k, the corners in the level's
// bins [w * kBinWindow, (w + 1) * kBinWindow); hist: one counter per bin of the window (dynamic
// LDS).
template <int P, int F>
__global__ __launch_bounds__(kBinThreads) void train_bin_count_kernel(TrainArgs t, BinMap bm,
                                                                      const float* __restrict__ in, uint32_t n,
                                                                      uint32_t* __restrict__ counts)
{
    extern __shared__ uint32_t hist[];
    constexpr uint32_t E = kBinFloats / F;
    const uint32_t k = blockIdx.y, w0 = blockIdx.z * kBinWindow, level_bins = bm.first[k + 1] - bm.first[k];
    if (w0 >= level_bins) return;
    const uint32_t first = bm.first[k] + w0, bins = level_bins - w0 < kBinWindow ? level_bins - w0 : kBinWindow;
    const GridLevel& lv = t.net.level[bm.level[k]];
    for (uint32_t j = threadIdx.x; j < bins; j += kBinThreads) hist[j] = 0u;
    __syncthreads();
    const uint32_t total = n * (uint32_t)P, j0 = blockIdx.x * kBinPairs;
    const uint32_t j1 = total - j0 < kBinPairs ? total : j0 + kBinPairs;
    for (uint32_t jj = j0 + threadIdx.x; jj < j1; jj += kBinThreads) {
        const uint32_t i = jj / P, p = jj - i * P;
        uint32_t idx[8];
        float fr[3];
        pair_corners<P>(lv, in, i, p, idx, fr);
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const uint32_t r = idx[c] / E - w0;
            if (r < bins) atomicAdd(&hist[r], 1u);
        }
    }
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < bins; j += kBinThreads)
        if (hist[j] != 0u) atomicAdd(&counts[first + j], hist[j]);
}

// One workgroup: offsets[b] = counts[0] + ... + counts[b - 1] for b <= bins, cursors = offsets.
__global__ __launch_bounds__(1024) void train_bin_scan_kernel(const uint32_t* __restrict__ counts, uint32_t bins,
                                                              uint32_t* __restrict__ offsets,
                                                              uint32_t* __restrict__ cursors)
{
    __shared__ uint32_t part[1024];
    const uint32_t tid = threadIdx.x, per = (bins + 1023u) / 1024u;
    const uint32_t b0 = tid * per < bins ? tid * per : bins, b1 = bins - b0 < per ? bins : b0 + per;
    uint32_t sum = 0;
    for (uint32_t b = b0; b < b1; b++) sum += counts[b];
    part[tid] = sum;
    __syncthreads();
    for (uint32_t off = 1; off < 1024u; off <<= 1) {
        const uint32_t v = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    uint32_t run = tid > 0 ? part[tid - 1] : 0u;
    for (uint32_t b = b0; b < b1; b++) {
        offsets[b] = run;
        cursors[b] = run;
        run += counts[b];
    }
    if (tid == 1023u) offsets[bins] = part[1023];
}

// The count kernel's workgroups again: local counts, a range of each touched bin reserved with one
// global atomic, then each term (entry within its bin, F values) written at the range's next
// position (LDS counter).
template <int P, int L, int F>
__global__ __launch_bounds__(kBinThreads) void train_bin_scatter_kernel(TrainArgs t, BinMap bm,
                                                                        const float* __restrict__ in,
                                                                        const float* __restrict__ act, uint32_t n,
                                                                        uint32_t* __restrict__ cursors,
                                                                        uint32_t* __restrict__ term_r,
                                                                        float* __restrict__ term_v)
{
    extern __shared__ uint32_t lds[];
    constexpr uint32_t E = kBinFloats / F;
    const uint32_t k = blockIdx.y, l = bm.level[k], w0 = blockIdx.z * kBinWindow;
    const uint32_t level_bins = bm.first[k + 1] - bm.first[k];
    if (w0 >= level_bins) return;
    const uint32_t first = bm.first[k] + w0, bins = level_bins - w0 < kBinWindow ? level_bins - w0 : kBinWindow;
    uint32_t* hist = lds;
    uint32_t* base = lds + bins;
    const GridLevel& lv = t.net.level[l];
    for (uint32_t j = threadIdx.x; j < bins; j += kBinThreads) hist[j] = 0u;
    __syncthreads();
    const uint32_t total = n * (uint32_t)P, j0 = blockIdx.x * kBinPairs;
    const uint32_t j1 = total - j0 < kBinPairs ? total : j0 + kBinPairs;
    for (uint32_t jj = j0 + threadIdx.x; jj < j1; jj += kBinThreads) {
        const uint32_t i = jj / P, p = jj - i * P;
        uint32_t idx[8];
        float fr[3];
        pair_corners<P>(lv, in, i, p, idx, fr);
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const uint32_t r = idx[c] / E - w0;
            if (r < bins) atomicAdd(&hist[r], 1u);
        }
    }
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < bins; j += kBinThreads) {
        const uint32_t c = hist[j];
        base[j] = c != 0u ? atomicAdd(&cursors[first + j], c) : 0u;
        hist[j] = 0u;
    }
    __syncthreads();
    const size_t S = t.act_stride;
    for (uint32_t jj = j0 + threadIdx.x; jj < j1; jj += kBinThreads) {
        const uint32_t i = jj / P, p = jj - i * P;
        uint32_t idx[8];
        float fr[3];
        pair_corners<P>(lv, in, i, p, idx, fr);
        float dx[F];
#pragma unroll
        for (int f = 0; f < F; f++) dx[f] = act[(size_t)(kDX + (p * L + l) * F + f) * S + i];
#pragma unroll
        for (uint32_t c = 0; c < 8; c++) {
            const uint32_t sl = idx[c] / E, r = sl - w0;
            if (r >= bins) continue;
            const uint32_t pos = base[r] + atomicAdd(&hist[r], 1u);
            const float w = corner_weight(c, fr);
            term_r[pos] = idx[c] - sl * E;
#pragma unroll
            for (int f = 0; f < F; f++) term_v[(size_t)pos * F + f] = w * dx[f];
        }
    }
}

// One workgroup per bin: the bin's terms added in LDS (kBinUnroll terms per thread loaded before
// their adds), the bin's entries stored whole (zeros included).
template <int F>
__global__ __launch_bounds__(kScatterThreads) void train_bin_accumulate_kernel(TrainArgs t, BinMap bm,
                                                                               const uint32_t* __restrict__ offsets,
                                                                               const uint32_t* __restrict__ term_r,
                                                                               const float* __restrict__ term_v,
                                                                               float* __restrict__ gtab)
{
    constexpr uint32_t E = kBinFloats / F;
    __shared__ float4 acc4[kBinFloats / 4];
    float* acc = reinterpret_cast<float*>(acc4);
    const uint32_t b = blockIdx.x;
    uint32_t k = 0;
    while (k + 1 < bm.count && b >= bm.first[k + 1]) k++;
    const GridLevel& lv = t.net.level[bm.level[k]];
    const uint32_t e0 = (b - bm.first[k]) * E;
    const uint32_t len = lv.size - e0 < E ? lv.size - e0 : E;  // a multiple of 8 entries
    for (uint32_t j = threadIdx.x; j < len * F / 4; j += kScatterThreads) acc4[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    const uint32_t q0 = offsets[b], q1 = offsets[b + 1];
    constexpr uint32_t U = kBinUnroll, B = kScatterThreads;
    for (uint32_t q = q0 + threadIdx.x; q < q1; q += U * B) {
        uint32_t r[U];
        float v[U][F];
#pragma unroll
        for (uint32_t h = 0; h < U; h++) {
            const uint32_t qq = q + h * B < q1 ? q + h * B : q;
            r[h] = term_r[qq];
#pragma unroll
            for (int f = 0; f < F; f++) v[h][f] = term_v[(size_t)qq * F + f];
        }
#pragma unroll
        for (uint32_t h = 0; h < U; h++) {
            if (q + h * B >= q1) break;
#pragma unroll
            for (int f = 0; f < F; f++) atomicAdd(&acc[r[h] * F + f], v[h][f]);
        }
    }
    __syncthreads();
    float4* out = reinterpret_cast<float4*>(gtab + ((size_t)lv.offset + e0) * F);
    for (uint32_t j = threadIdx.x; j < len * F / 4; j += kScatterThreads) out[j] = acc4[j];
}

// Partial dW[o][k] = sum over samples b in [b0, b1) of delta_b[o] * act_b[k] for one matrix (O
// outputs, I inputs), b ascending: tiles of 32 samples of the O delta rows and the I activation rows
// are staged in LDS (sm, (O + I) x 33 floats); the 32 x 32 blocks of the matrix go round the
// workgroup's 4 waves, each block a chain of v_mfma_f32_32x32x2_f32 over the samples.
// Measured per 65,536 samples (all five matrices): 44 us; 92 us with FMAs on LDS operands, and 91
// on the matrix cores without the next tile's loads in flight.
template <int O, int I>
__device__ __forceinline__ void wgrad_chunk(const float* __restrict__ act, size_t S, int d_row, int a_row, uint32_t b0,
                                            uint32_t b1, float* sm, float* __restrict__ out)
{
    constexpr int RB = (O + 31) / 32, CB = I / 32, BLOCKS = RB * CB, PER = (BLOCKS + 3) / 4;
    static_assert(I % 32 == 0 && (O % 32 == 0 || O < 32), "blocks of 32 x 32");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, c = lane & 31;
    floatx16_t acc[PER] = {};
    // Four samples of a row per load (rows and chunks start at multiples of 32 samples; a row has
    // at least the samples up to the next multiple of 32); the next tile is loaded while this
    // one is multiplied.
    constexpr int QUADS = (O + I) * 8, LOADS = (QUADS + 255) / 256;
    float4 v[LOADS];
    auto load = [&](uint32_t c0) {
#pragma unroll
        for (int m = 0; m < LOADS; m++) {
            const int e = tid + m * 256, r = e >> 3;
            const int src = r < O ? d_row + r : a_row + (r - O);
            if (e < QUADS) v[m] = *reinterpret_cast<const float4*>(act + (size_t)src * S + c0 + 4 * (e & 7));
        }
    };
    if (b0 < b1) load(b0);
    for (uint32_t c0 = b0; c0 < b1; c0 += 32) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < LOADS; m++) {
            const int e = tid + m * 256;
            if (e < QUADS) {
                const uint32_t b = c0 + 4 * (e & 7);
                float* d = sm + (e >> 3) * 33 + 4 * (e & 7);
                d[0] = b < b1 ? v[m].x : 0.f;
                d[1] = b + 1 < b1 ? v[m].y : 0.f;
                d[2] = b + 2 < b1 ? v[m].z : 0.f;
                d[3] = b + 3 < b1 ? v[m].w : 0.f;
            }
        }
        __syncthreads();
        if (c0 + 32 < b1) load(c0 + 32);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int blk = wave + 4 * q;
            if (blk < BLOCKS) {
                // Rows past O (the 8-output matrix) repeat its rows; their products are not stored.
                const float* d = sm + ((blk / CB) * 32 + c) % O * 33 + g;
                const float* x = sm + (O + (blk % CB) * 32 + c) * 33 + g;
#pragma unroll
                for (int s = 0; s < 16; s++)
                    acc[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(d[2 * s], x[2 * s], acc[q], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int blk = wave + 4 * q;
        if (blk < BLOCKS) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int o = (blk / CB) * 32 + 8 * (r / 4) + 4 * g + r % 4;
                if (o < O) out[o * I + (blk % CB) * 32 + c] = acc[q][r];
            }
        }
    }
}

// Workgroup (chunk c, matrix l): the partial of samples [c * per, min(n, (c + 1) * per)).
__global__ __launch_bounds__(256) void train_wgrad_kernel(const float* __restrict__ act, uint32_t S, uint32_t n,
                                                          uint32_t per, float* __restrict__ part)
{
    __shared__ float sm[(kH + kK0) * 33];
    const int layer = blockIdx.y;
    const uint32_t b0 = blockIdx.x * per, b1 = b0 + per < n ? b0 + per : n;
    float* out = part + (size_t)blockIdx.x * kMlp + w_offset(layer);
    if (layer == 0)
        wgrad_chunk<kH, kK0>(act, S, kD, kA0, b0, b1, sm, out);
    else if (layer == 4)
        wgrad_chunk<kO, kH>(act, S, kD5, kHid + 3 * kH, b0, b1, sm, out);
    else
        wgrad_chunk<kH, kH>(act, S, kD + layer * kH, kHid + (layer - 1) * kH, b0, b1, sm, out);
}

// grad[j] = sum of the chunks' partials: eight running sums over chunks c = r mod 8 (eight loads in
// flight per thread), added in a fixed order, so the result does not depend on the schedule. The
// workgroup past the matrix entries adds the n_losses losses of the backward pass, in double: lane
// t those of t, t + 64, ... in order, then the lanes pairwise.
__global__ __launch_bounds__(64) void train_wgrad_reduce_kernel(const float* __restrict__ part, uint32_t chunks,
                                                                float* __restrict__ grad,
                                                                const double* __restrict__ losses, uint32_t n_losses,
                                                                float* __restrict__ loss)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= kMlp) {
        static_assert(kMlp % 64 == 0, "the last workgroup has no matrix entries");
        double s = 0.0;
        for (uint32_t k = threadIdx.x; k < n_losses; k += 64u) s += losses[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (threadIdx.x == 0) *loss = (float)s;
        return;
    }
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    uint32_t c = 0;
    for (; c + 8 <= chunks; c += 8) {
#pragma unroll
        for (int r = 0; r < 8; r++) s[r] += part[(size_t)(c + r) * kMlp + j];
    }
    for (; c < chunks; c++) s[0] += part[(size_t)c * kMlp + j];
    grad[j] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// tiny-cuda-nn's AdamOptimizer step (public optimizers/adam.h, the reference's optimiser):
// MATRIX parameters (the MLP) get L2 regularisation added to the gradient and are updated every
// step, also with a zero gradient (their moments decay); the other parameters (the grid tables)
// are skipped where the gradient is exactly zero and get no L2 term. Each parameter counts its
// own updates t, and the bias correction is folded into the rate:
// w -= lr * sqrt(1 - beta2^t) / (1 - beta1^t) * m / (sqrt(v) + epsilon).
template <bool MATRIX>
__global__ __launch_bounds__(256) void train_adam_kernel(float* __restrict__ w, const float* __restrict__ g,
                                                         float* __restrict__ m, float* __restrict__ v,
                                                         uint32_t* __restrict__ steps, uint64_t n, AdamArgs h)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gi = g[i];
    if (MATRIX)
        gi += h.l2_reg * w[i];
    else if (gi == 0.f)
        return;  // sparse update: entries no sample touched keep their value, moments and count
    const float mi = h.beta1 * m[i] + (1.f - h.beta1) * gi;
    const float vi = h.beta2 * v[i] + (1.f - h.beta2) * gi * gi;
    const uint32_t t = steps[i] + 1u;
    const float lr = h.lr * sqrtf(1.f - powf(h.beta2, (float)t)) / (1.f - powf(h.beta1, (float)t));
    m[i] = mi;
    v[i] = vi;
    steps[i] = t;
    w[i] = w[i] - lr * mi / (sqrtf(vi) + h.epsilon);
}

__global__ __launch_bounds__(256) void train_zero_kernel(float* __restrict__ p, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}

}  // namespace dev

uint32_t train_act_stride(uint32_t max_batch) { return (max_batch + 63u) & ~63u; }

size_t train_act_bytes(uint32_t max_batch)
{
    const size_t stride = train_act_stride(max_batch);
    return (dev::kRows * stride + (size_t)dev::kMlp * (2 + dev::kChunks)) * sizeof(float) +
           stride / dev::kMinGroup * sizeof(double);
}

hipError_t train_zero(float* p, uint64_t n, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(dev::train_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, p, n);
    return hipGetLastError();
}

// Bin workspace: the bin counts, offsets and cursors, then the corner terms of a max batch
// (P * L * 8 per sample: entry within its slice, and F values).
constexpr uint32_t kMaxBins = 131072;  // bins of all binned levels (2^26 entries x 16 levels at 2 features)

size_t train_bin_bytes(uint32_t max_batch, uint32_t n_points, uint32_t n_levels, uint32_t n_features)
{
    const size_t terms = (size_t)train_act_stride(max_batch) * n_points * n_levels * 8u;
    return (size_t)3 * (kMaxBins + 1) * sizeof(uint32_t) + terms * (1 + n_features) * sizeof(float);
}

// The caller guarantees n <= act_stride (the trainer's max batch).
hipError_t train_gradients(const TrainArgs& t, const float* in, const float* targets, uint32_t n, hipStream_t stream,
                           bool* supported)
{
    *supported = true;
    if (n == 0) return hipSuccess;
    if (n > t.act_stride) return hipErrorInvalidValue;
    const NetArgs& a   = t.net;
    const size_t   S   = t.act_stride;
    float* const   act = t.act;
    float* const   wf  = act + (size_t)dev::kRows * S;  // rows of a multiple of 64 floats: 16-byte aligned
    float* const   wb  = wf + dev::kMlp;
    float* const   part = wb + dev::kMlp;
    double* const  losses = reinterpret_cast<double*>(part + (size_t)dev::kMlp * dev::kChunks);
    const dim3 grid_mlp((dev::kMlp + 255) / 256);
    const bool small = n <= dev::kSmallBatch;
    const uint32_t per_wg = (small ? 2u : 8u) * dev::kWaveSamples;
    const dim3 grid((n + per_wg - 1) / per_wg), block((small ? 2u : 8u) * 64u);
    if (a.n_levels > (uint32_t)kMaxLevels || a.n_features == 0) return hipErrorInvalidValue;
    // Levels of at least NBVH_BIN_MIN_SLICES slices (16 MB of gradient) take the binned path; the
    // others are scanned once per slice, split into parts so that each workgroup adds about 32K
    // corners if the batch's corners spread evenly over the level (a skewed batch only makes some
    // workgroups slower). Measured per 65,536-sample step of the 16 x 2 grid, binning levels of
    // >= 16 / 64 / 128 slices and slice scans only (2048 pairs per binning workgroup): 2^19 1.14 /
    // 1.06 / 1.06 / 1.06 ms, 2^20 1.37 / 1.40 / 1.32 / 1.32, 2^21 1.66 / 1.69 / 1.69 / 1.89, 2^22
    // 2.06 / 2.09 / 2.09 / 2.74, 2^23 2.60 / 2.62 / 2.62 / 4.03 (global atomics on the gradient,
    // the earlier form for the largest tables: 2^22 2.82, 2^23 3.83), all with one thread per sample
    // in both passes. On the matrix cores, with 128: 0.81 / 1.09 / 1.37 / 1.73 / 2.27 ms.
#ifndef NBVH_BIN_MIN_SLICES
#define NBVH_BIN_MIN_SLICES 128
#endif
    dev::SliceMap map{};
    dev::BinMap bins{};
    uint32_t max_bins = 0;
    for (uint32_t l = 0; l < a.n_levels; l++) {
        const uint32_t E = dev::kSliceFloats / a.n_features, size = a.level[l].size;
        const uint32_t slices = (size + E - 1) / E;
        const double corners = (double)n * a.n_points * 8.0 * std::min(E, size) / size;
        if (slices >= NBVH_BIN_MIN_SLICES) {
            const uint32_t EB = dev::kBinFloats / a.n_features, level_bins = (size + EB - 1) / EB;
            map.parts[l]     = 1;
            map.first[l + 1] = map.first[l];
            bins.level[bins.count]     = l;
            bins.first[bins.count + 1] = bins.first[bins.count] + level_bins;
            bins.count++;
            max_bins = std::max(max_bins, level_bins);
            continue;
        }
        map.parts[l]     = (uint32_t)std::min(64.0, std::max(1.0, std::ceil(corners / 32768.0)));
        map.first[l + 1] = map.first[l] + slices * map.parts[l];
    }
    const uint32_t n_bins = bins.first[bins.count];
    if (n_bins > kMaxBins) return hipErrorInvalidValue;
    // Term positions are 32-bit: a step bins fewer than 2^32 corner terms.
    if ((uint64_t)n * a.n_points * 8u * bins.count > 0xFFFFFFFFull) return hipErrorInvalidValue;
    const uint32_t windows = (max_bins + dev::kBinWindow - 1) / dev::kBinWindow;
    const uint32_t window_bins = std::min(max_bins, dev::kBinWindow);
    uint32_t* const counts  = reinterpret_cast<uint32_t*>(t.bins);
    uint32_t* const offsets = counts + (kMaxBins + 1);
    uint32_t* const cursors = offsets + (kMaxBins + 1);
    uint32_t* const term_r  = cursors + (kMaxBins + 1);
    float* const    term_v  = reinterpret_cast<float*>(term_r + (size_t)S * a.n_points * a.n_levels * 8u);
    const dim3 bin_grid((n * a.n_points + dev::kBinPairs - 1) / dev::kBinPairs, bins.count, windows);
    // Split slices add into the gradient with global atomics: their levels start from zero, one
    // launch for each run of them. Every other entry is stored by its slice.
    for (uint32_t l = 0; l < a.n_levels;) {
        if (map.parts[l] <= 1) {
            l++;
            continue;
        }
        const uint32_t first = a.level[l].offset;
        uint64_t end = first;
        for (; l < a.n_levels && map.parts[l] > 1; l++) end = (uint64_t)a.level[l].offset + a.level[l].size;
        const hipError_t e =
            train_zero(t.grad_tables + (size_t)first * a.n_features, (end - first) * a.n_features, stream);
        if (e != hipSuccess) return e;
    }
    if (n_bins > 0) {
        const hipError_t e = train_zero(reinterpret_cast<float*>(counts), n_bins, stream);
        if (e != hipSuccess) return e;
    }
    bool shape = false;
#define X(P_, L_, F_)                                                                                                \
    if (a.n_points == P_ && a.n_levels == L_ && a.n_features == F_) {                                                \
        shape = true;                                                                                                \
        hipLaunchKernelGGL(dev::train_fragments_kernel, grid_mlp, dim3(256), 0, stream, t.mlp, wf, wb);              \
        if (small)                                                                                                   \
            hipLaunchKernelGGL((dev::train_forward_kernel<P_, L_, F_, 2>), grid, block, 0, stream, t,                \
                               (const float*)wf, in, act, n);                                                        \
        else                                                                                                         \
            hipLaunchKernelGGL((dev::train_forward_kernel<P_, L_, F_, 8>), grid, block, 0, stream, t,                \
                               (const float*)wf, in, act, n);                                                        \
        if (small)                                                                                                   \
            hipLaunchKernelGGL(dev::train_backward_kernel<2>, grid, block, 0, stream, t, (const float*)wb, targets,  \
                               act, losses, n);                                                                      \
        else                                                                                                         \
            hipLaunchKernelGGL(dev::train_backward_kernel<8>, grid, block, 0, stream, t, (const float*)wb, targets,  \
                               act, losses, n);                                                                      \
        if (map.first[L_] > 0)                                                                                       \
            hipLaunchKernelGGL((dev::train_scatter_kernel<P_, L_, F_>), dim3(map.first[L_]), dim3(dev::kScatterThreads), \
                               0, stream, t, map, in, (const float*)act, t.grad_tables, n);                          \
        if (n_bins > 0) {                                                                                            \
            hipLaunchKernelGGL((dev::train_bin_count_kernel<P_, F_>), bin_grid, dim3(dev::kBinThreads),                \
                               window_bins * 4, stream, t, bins, in, n, counts);                                     \
            hipLaunchKernelGGL(dev::train_bin_scan_kernel, dim3(1), dim3(1024), 0, stream, (const uint32_t*)counts,  \
                               n_bins, offsets, cursors);                                                           \
            hipLaunchKernelGGL((dev::train_bin_scatter_kernel<P_, L_, F_>), bin_grid, dim3(dev::kBinThreads),          \
                               window_bins * 8, stream, t, bins, in, (const float*)act, n, cursors, term_r, term_v);  \
            hipLaunchKernelGGL((dev::train_bin_accumulate_kernel<F_>), dim3(n_bins), dim3(dev::kScatterThreads), 0,   \
                               stream, t, bins, (const uint32_t*)offsets, (const uint32_t*)term_r,                  \
                               (const float*)term_v, t.grad_tables);                                                \
        }                                                                                                            \
    }
    X(3, 16, 2) X(3, 8, 4)
#undef X
    if (!shape) {
        *supported = false;
        return hipSuccess;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // Chunks of a multiple of 32 samples, at most kChunks of them.
    const uint32_t target = std::min<uint32_t>(dev::kChunks, (n + 255) / 256);
    const uint32_t per = ((n + target - 1) / target + 31u) & ~31u, chunks = (n + per - 1) / per;
    hipLaunchKernelGGL(dev::train_wgrad_kernel, dim3(chunks, dev::kLayers), dim3(256), 0, stream, (const float*)act,
                       (uint32_t)S, n, per, part);
    hipLaunchKernelGGL(dev::train_wgrad_reduce_kernel, dim3(dev::kMlp / 64 + 1), dim3(64), 0, stream,
                       (const float*)part, chunks, t.grad_mlp, (const double*)losses, grid.x, t.loss);
    return hipGetLastError();
}

hipError_t train_adam(float* w, const float* g, float* m, float* v, uint32_t* steps, uint64_t n, bool matrix,
                      const AdamArgs& h, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (matrix)
        hipLaunchKernelGGL(dev::train_adam_kernel<true>, grid, dim3(256), 0, stream, w, g, m, v, steps, n, h);
    else
        hipLaunchKernelGGL(dev::train_adam_kernel<false>, grid, dim3(256), 0, stream, w, g, m, v, steps, n, h);
    return hipGetLastError();
}

}  // namespace nbvh
