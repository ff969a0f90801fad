// neural_fp32.hip -- the FP32 neural query (FP32 hash tables, FP32 matrix cores) and the FP32
// network inference. One wave evaluates the 64 segments of its slots: every lane gathers its own
// segment's features, the MLP runs on v_mfma_f32_32x32x2_f32 (device/mlp_f32.h).
//
// Arithmetic order is that of oracle/nbvh_oracle.cpp (FP32 mode): the FP32 path is bit-exact
// with it.
#include <hip/hip_runtime.h>

#include "../device/mlp_f32.h"
#include "../device/wave_query.h"
#include "launch.h"

namespace nbvh {
namespace dev {

// One workgroup of 8 waves per CU (two per SIMD) shares one LDS copy of the weights (74 KB for 96
// inputs); with the waves' stacks (48 KB) and the node cache (16 KB) it takes 138 of 160 KB.
constexpr int kF32Waves = 8;

template <int P, int L, int F, bool PARTS, int ND, Gather G>
__global__ __launch_bounds__(64 * kF32Waves, 2) void neural_query_fp32_kernel(NetArgs a, RayBatch b,
                                                                             uint32_t* __restrict__ queue)
{
    constexpr int K0 = P * L * F;
    __shared__ float4 w_lds[F32Layout<K0>::FLOATS / 4];
    __shared__ uint32_t stack_lds[kF32Waves * kNeuralStackSize * 64];
    __shared__ uint4 node_lds[2 * kNodeCache];
    const uint32_t n_cached = stage_nodes(a, node_lds);
    stage_weights_f32<K0>(a.mlp_f32, w_lds);
    __syncthreads();
    const CachedNodes nodes{a.nodes, node_lds, n_cached};
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    LdsStack st{stack_lds + wave * kNeuralStackSize * 64 + lane, 0};
    RayQueue q;
    q.init(queue, batch_count(b), a.image_width, a.queue_bands);
    Slot s;
    const uint32_t slots = first_rays<PARTS>(a, b, q, s);
    while (fill_slots<PARTS>(a, nodes, s, st, b, q)) {
        float x[K0];
        if constexpr (G == Gather::WIDE) {
            float pts[3 * P];
#pragma unroll
            for (int c = 0; c < 3 * P; c++) pts[c] = 0.5f;
            if (s.state == SLOT_SEG) encode_segment(a, s.ray, s.seg_mint, s.seg_maxt, pts, &s.rng);
            gather_wide_f32<P, L, F>(a, a.tables_f32, slots, pts, x);
        } else if (s.state == SLOT_SEG) {
            float pts[3 * P];
            encode_segment(a, s.ray, s.seg_mint, s.seg_maxt, pts, &s.rng);
            wave_features_f32<P, L, F, ND, G>(a, a.tables_f32, pts, x);
        } else {
#pragma unroll
            for (int k = 0; k < K0; k++) x[k] = 0.f;
        }
        // WIDE: at most 32 slots, the second block of 32 segments is empty.
        float z[8];
        mlp_wave_f32<K0, G == Gather::WIDE ? 1 : 2>(reinterpret_cast<const float*>(w_lds), x, z);
        if (s.state == SLOT_SEG) consume_segment<PARTS>(a, s, z, b);
    }
}

// tcnn::Network::inference replacement, FP32: in[n x 3P] -> out[n x 8] (sigmoid), logits.
// Persistent over chunks of `group` inputs, a multiple of 64 up to blockDim.x (network_waves), so
// that every lane of a working wave takes part in each MFMA; the weights are staged once per
// workgroup, by all its waves.
template <int P, int L, int F, int ND>
__global__ __launch_bounds__(64 * kF32Waves, 2) void network_fp32_kernel(NetArgs a, const float* __restrict__ in,
                                                                        uint32_t n, uint32_t group,
                                                                        float* __restrict__ out,
                                                                        float* __restrict__ logits)
{
    constexpr int K0 = P * L * F;
    __shared__ float4 w_lds[F32Layout<K0>::FLOATS / 4];
    stage_weights_f32<K0>(a.mlp_f32, w_lds);
    __syncthreads();
    if (threadIdx.x >= group) return;
    for (uint32_t base = blockIdx.x * group; base < n; base = next_chunk(base, group, n)) {
        asm volatile("" ::: "memory");  // keeps the weights' LDS reads in the loop (hoisted, they spill)
        const uint32_t i = base + threadIdx.x;
        float x[K0];
        if (i < n) {
            float pts[3 * P];
#pragma unroll
            for (int c = 0; c < 3 * P; c++) pts[c] = in[(size_t)i * (3 * P) + c];
            wave_features_f32<P, L, F, ND, Gather::LEVELS>(a, a.tables_f32, pts, x);
        } else {
#pragma unroll
            for (int k = 0; k < K0; k++) x[k] = 0.f;
        }
        float z[8];
        mlp_wave_f32<K0, 2>(reinterpret_cast<const float*>(w_lds), x, z);
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

template <int P, int L, int F, bool PARTS>
static hipError_t launch_fp32_query_k(const NetArgs& a, const RayBatch& rb, uint32_t* queue, uint32_t n_cus,
                                      hipStream_t stream, QueryGrid* plan)
{
    using dev::Gather;
    constexpr uint32_t threads = 64 * dev::kF32Waves;
    auto k = dev::neural_query_fp32_kernel<P, L, F, PARTS, -1, Gather::LEVELS>;
    static const uint32_t bpc = blocks_per_cu(k, threads);
    const uint32_t cap = a.blocks_per_cu != 0u && a.blocks_per_cu < bpc ? a.blocks_per_cu : bpc;
    const QueryGrid g = query_grid(rb, dev::kF32Waves, n_cus * cap, 64u / L < 16u ? 64u / L : 16u, 32u);
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
    if (g.wide) {
        k = dev::neural_query_fp32_kernel<P, L, F, PARTS, -1, Gather::WIDE>;
    } else if constexpr (L > kDensePrefix) {
        // The hash-only gather for grids whose levels from the 4th on are hashed (the two
        // benchmark shapes); other grids take the general gather.
        if (a.n_dense == (uint32_t)kDensePrefix)
            k = dev::neural_query_fp32_kernel<P, L, F, PARTS, kDensePrefix, dev::kQueryGather<L, kDensePrefix>>;
    }
    hipLaunchKernelGGL(k, dim3(g.blocks), dim3(threads), 0, stream, args, rb, queue);
    return hipGetLastError();
}

template <int P, int L, int F>
static hipError_t launch_fp32_query(const NetArgs& a, const RayBatch& rb, uint32_t* queue, uint32_t n_cus,
                                    hipStream_t stream, QueryGrid* plan)
{
    return rb.parts ? launch_fp32_query_k<P, L, F, true>(a, rb, queue, n_cus, stream, plan)
                    : launch_fp32_query_k<P, L, F, false>(a, rb, queue, n_cus, stream, plan);
}

template <int P, int L, int F, int ND>
static hipError_t launch_fp32_network_k(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits,
                                        uint32_t n_cus, hipStream_t stream)
{
    auto k = dev::network_fp32_kernel<P, L, F, ND>;
    constexpr uint32_t threads = 64 * dev::kF32Waves;
    static const uint32_t bpc = blocks_per_cu(k, threads);
    const uint32_t resident = n_cus * bpc, group = 64u * network_waves(n, dev::kF32Waves, resident);
    uint32_t blocks = n / group + (n % group != 0u ? 1u : 0u);
    blocks = blocks < resident ? blocks : resident;
    hipLaunchKernelGGL(k, dim3(blocks), dim3(threads), 0, stream, a, in, n, group, out, logits);
    return hipGetLastError();
}

template <int P, int L, int F>
static hipError_t launch_fp32_network(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits,
                                      uint32_t n_cus, hipStream_t stream)
{
    if constexpr (L > kDensePrefix) {
        if (a.n_dense == (uint32_t)kDensePrefix)
            return launch_fp32_network_k<P, L, F, kDensePrefix>(a, in, n, out, logits, n_cus, stream);
    }
    return launch_fp32_network_k<P, L, F, -1>(a, in, n, out, logits, n_cus, stream);
}

#define NBVH_FP32_SHAPES(X) X(3, 16, 2) X(3, 8, 4) X(3, 2, 2) X(3, 4, 2)

hipError_t query_fp32(const NetArgs& a, const RayBatch& rb, uint32_t* queue, uint32_t n_cus, hipStream_t stream,
                      bool* supported, QueryGrid* plan)
{
    *supported = true;
#define X(P_, L_, F_)                                                                                    \
    if (a.n_points == P_ && a.n_levels == L_ && a.n_features == F_ && a.n_hidden_layers == 4)            \
        return launch_fp32_query<P_, L_, F_>(a, rb, queue, n_cus, stream, plan);
    NBVH_FP32_SHAPES(X)
#undef X
    *supported = false;
    return hipSuccess;
}

hipError_t network_fp32(const NetArgs& a, const float* in, uint32_t n, float* out, float* logits,
                        uint32_t n_cus, hipStream_t stream, bool* supported)
{
    *supported = true;
#define X(P_, L_, F_)                                                                                    \
    if (a.n_points == P_ && a.n_levels == L_ && a.n_features == F_ && a.n_hidden_layers == 4)            \
        return launch_fp32_network<P_, L_, F_>(a, in, n, out, logits, n_cus, stream);
    NBVH_FP32_SHAPES(X)
#undef X
    *supported = false;
    return hipSuccess;
}

}  // namespace nbvh
