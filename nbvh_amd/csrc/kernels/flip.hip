// flip.hip -- LDR-FLIP image error of a rendering against a reference rendering, the metric of the
// reference's validation mode (compute_and_display_flip_error,
// src/cuda/neural/neural_bvh_renderer.cu:40-92), written from the published method (Andersson et
// al., "FLIP: A Difference Evaluator for Alternating Images", HPG 2020) with the steps and
// constants of the method's reference implementation (figures/flip/flip_api.py:439-497):
//
//   flip_prepare_kernel  per pixel of both accumulation buffers (rgb sum, sample count): mean
//                        linear RGB -> sRGB clamped to [0, 1] -> linear RGB -> YyCxCz and Y / Yn;
//   flip_error_kernel    32 x 16 pixel tiles with a halo of the larger kernel radius in LDS
//                        (edge pixels replicated): the contrast-sensitivity filtered YyCxCz of both
//                        images -> linear RGB clamped -> CIELab -> Hunt -> HyAB^0.7 remapped (colour
//                        error); edge and point responses of Y / Yn (feature error); the pixel's
//                        error dEc^(1 - dEf); per-tile sums of the errors;
//   flip_mean_kernel     the tile sums added in a fixed order (one workgroup), / pixel count.
// Every filter is a sum of products of 1D profiles (the sensitivity kernels are one or two
// Gaussians, the detectors a derivative profile along one axis and a Gaussian along the other), so
// each tile is filtered along x, then along y, in LDS: 7 + 8 profiles of 2 r + 1 taps per pixel
// and image instead of 3 (2 rc + 1)^2 + 4 (2 rf + 1)^2 taps. The profiles are computed on the host
// (FP64, rounded to FP32). FP32 arithmetic. The rate is set by the LDS reads of the two passes.
// Measured at 1920 x 1080, the whole call: 247 us; with 2D filters (2088 us), a one-thread mean
// (433) and the sRGB encoding and decoding in the prepare step (93) 2709 us.
#include <hip/hip_runtime.h>

#include "../nbvh_internal.h"
#include "launch.h"

namespace nbvh {
namespace dev {

constexpr int kFlipTileX = 32, kFlipTileY = 16;
constexpr int kFlipThreads = kFlipTileX * kFlipTileY;  // one pixel per thread

// XYZ of linear sRGB (D65 primaries) normalised by the illuminant (times its reciprocal).
__device__ __forceinline__ void rgb_to_xyz_n(const FlipArgs& a, const float rgb[3], float xyz[3])
{
    for (int r = 0; r < 3; r++)
        xyz[r] = (a.rgb2xyz[3 * r] * rgb[0] + a.rgb2xyz[3 * r + 1] * rgb[1] + a.rgb2xyz[3 * r + 2] * rgb[2]) * a.inv_white[r];
}

__device__ __forceinline__ float lab_f(float t)
{
    const float d = 6.f / 29.f;
    return t > d * d * d ? cbrtf(t) : t / (3.f * d * d) + 4.f / 29.f;
}

// Hunt-adjusted CIELab of a YyCxCz colour after conversion to linear RGB clamped to [0, 1].
__device__ __forceinline__ void ycc_to_hunt_lab(const FlipArgs& a, const float ycc[3], float lab[3])
{
    const float y = (ycc[0] + 16.f) / 116.f;
    const float xyz[3] = {(ycc[1] / 500.f + y) * a.white[0], y * a.white[1], (y - ycc[2] / 200.f) * a.white[2]};
    float rgb[3];
    for (int r = 0; r < 3; r++) {
        const float v = a.xyz2rgb[3 * r] * xyz[0] + a.xyz2rgb[3 * r + 1] * xyz[1] + a.xyz2rgb[3 * r + 2] * xyz[2];
        rgb[r] = fminf(fmaxf(v, 0.f), 1.f);
    }
    float n[3];
    rgb_to_xyz_n(a, rgb, n);
    const float fx = lab_f(n[0]), fy = lab_f(n[1]), fz = lab_f(n[2]);
    const float L = 116.f * fy - 16.f;
    lab[0] = L;
    lab[1] = 0.01f * L * (500.f * (fx - fy));
    lab[2] = 0.01f * L * (200.f * (fy - fz));
}

__global__ __launch_bounds__(256) void flip_prepare_kernel(FlipArgs a)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.w * a.h) return;
    for (int img = 0; img < 2; img++) {
        const float4 acc = reinterpret_cast<const float4*>(img == 0 ? a.ref : a.test)[i];
        float rgb[3] = {0.f, 0.f, 0.f};
        if (acc.w > 0.f) {
            rgb[0] = acc.x / acc.w;
            rgb[1] = acc.y / acc.w;
            rgb[2] = acc.z / acc.w;
        }
        // LDR-FLIP takes sRGB clamped to [0, 1] and decodes it again: encoding and decoding are
        // inverse and monotonic on [0, 1], so the clamp alone is the exact value of the three.
        for (int c = 0; c < 3; c++) rgb[c] = fminf(fmaxf(rgb[c], 0.f), 1.f);
        float n[3];
        rgb_to_xyz_n(a, rgb, n);
        reinterpret_cast<float4*>(img == 0 ? a.prep_ref : a.prep_test)[i] =
            make_float4(116.f * n[1] - 16.f, 500.f * (n[0] - n[1]), 200.f * (n[1] - n[2]), n[1]);
    }
}

// Filtered values of one image at this thread's pixel: f = YyCxCz after the sensitivity kernels,
// edge and point magnitudes. tile: the prepared image, (X + 2r) x (Y + 2r) pixels; hx: the seven
// x-filtered planes of its (Y + 2r) rows.
__device__ __forceinline__ void flip_filter(const FlipArgs& a, const float4* tile, float* hx, float f[3], float& edge,
                                            float& point)
{
    const int r = a.r, TW = kFlipTileX + 2 * r, rows = kFlipTileY + 2 * r, plane = rows * kFlipTileX;
    for (int k = threadIdx.x; k < plane; k += kFlipThreads) {
        const float4* row = tile + (k / kFlipTileX) * TW + k % kFlipTileX;
        const float yc = row[r].w;
        float s[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int t = 0; t <= 2 * r; t++) {
            const float4 v = row[t];
            const FlipTap w = a.taps[t];
            s[0] = fmaf(w.achromatic, v.x, s[0]);
            s[1] = fmaf(w.red_green, v.y, s[1]);
            s[2] = fmaf(w.blue_yellow[0], v.z, s[2]);
            s[3] = fmaf(w.blue_yellow[1], v.z, s[3]);
            // The detectors' profiles sum to zero, so they are applied to Y - Y(centre): the same
            // responses, without the rounding residue of the weights' sum times Y, which the
            // square root of the feature error would magnify on flat regions.
            s[4] = fmaf(w.smooth, v.w, s[4]);
            s[5] = fmaf(w.edge, v.w - yc, s[5]);
            s[6] = fmaf(w.point, v.w - yc, s[6]);
        }
#pragma unroll
        for (int c = 0; c < 7; c++) hx[c * plane + k] = s[c];
    }
    __syncthreads();
    const float* col = hx + threadIdx.x;  // pixel (tx, ty): rows ty .. ty + 2 r of column tx
    const float gc = col[4 * plane + r * kFlipTileX];
    float by[2] = {0.f, 0.f}, ex = 0.f, ey = 0.f, qx = 0.f, qy = 0.f;
    f[0] = f[1] = 0.f;
    for (int t = 0; t <= 2 * r; t++) {
        const float* v = col + t * kFlipTileX;
        const FlipTap w = a.taps[t];
        f[0]  = fmaf(w.achromatic, v[0], f[0]);
        f[1]  = fmaf(w.red_green, v[plane], f[1]);
        by[0] = fmaf(w.blue_yellow[0], v[2 * plane], by[0]);
        by[1] = fmaf(w.blue_yellow[1], v[3 * plane], by[1]);
        const float g = v[4 * plane] - gc;
        ey = fmaf(w.edge, g, ey);
        qy = fmaf(w.point, g, qy);
        ex = fmaf(w.smooth, v[5 * plane], ex);
        qx = fmaf(w.smooth, v[6 * plane], qx);
    }
    f[2]  = fmaf(a.by_weight[0], by[0], a.by_weight[1] * by[1]);
    edge  = sqrtf(ex * ex + ey * ey);
    point = sqrtf(qx * qx + qy * qy);
    __syncthreads();
}

__global__ __launch_bounds__(kFlipThreads) void flip_error_kernel(FlipArgs a)
{
    extern __shared__ float4 lds[];
    __shared__ double sums[kFlipThreads];
    const int r = a.r, TW = kFlipTileX + 2 * r, TH = kFlipTileY + 2 * r;
    float* hx = reinterpret_cast<float*>(lds + TW * TH);
    const int tx = threadIdx.x % kFlipTileX, ty = threadIdx.x / kFlipTileX;
    const int x0 = blockIdx.x * kFlipTileX, y0 = blockIdx.y * kFlipTileY;
    const int W = (int)a.w, H = (int)a.h;
    float lab[2][3], edge[2], point[2];
#pragma unroll
    for (int img = 0; img < 2; img++) {
        const float4* src = reinterpret_cast<const float4*>(img == 0 ? a.prep_ref : a.prep_test);
        for (int k = threadIdx.x; k < TW * TH; k += kFlipThreads) {
            const int gx = min(max(x0 + k % TW - r, 0), W - 1), gy = min(max(y0 + k / TW - r, 0), H - 1);
            lds[k] = src[(size_t)gy * W + gx];
        }
        __syncthreads();
        float f[3];
        flip_filter(a, lds, hx, f, edge[img], point[img]);
        ycc_to_hunt_lab(a, f, lab[img]);
    }
    const int px = x0 + tx, py = y0 + ty;
    float err = 0.f;
    if (px < W && py < H) {
        const float dl = fabsf(lab[0][0] - lab[1][0]);
        const float da = lab[0][1] - lab[1][1], db = lab[0][2] - lab[1][2];
        float dec = powf(dl + sqrtf(da * da + db * db), 0.7f);
        const float pcm = 0.4f * a.cmax;
        dec = dec < pcm ? (0.95f / pcm) * dec : 0.95f + (dec - pcm) / (a.cmax - pcm) * 0.05f;
        const float fd = fmaxf(fabsf(edge[0] - edge[1]), fabsf(point[0] - point[1])) * 0.70710678118654752f;
        const float def = sqrtf(fd);
        err = powf(dec, 1.f - def);
        if (a.map) a.map[(size_t)py * W + px] = err;
    }
    sums[threadIdx.x] = (double)err;
    __syncthreads();
    for (int s = kFlipThreads / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sums[threadIdx.x] += sums[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.partials[blockIdx.y * gridDim.x + blockIdx.x] = sums[0];
}

// Thread t adds the partials t, t + 1024, ... in order, then the threads' sums pairwise.
__global__ __launch_bounds__(1024) void flip_mean_kernel(const double* __restrict__ partials, uint32_t n, double pixels,
                                                         double* __restrict__ out)
{
    __shared__ double sums[1024];
    double s = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += 1024u) s += partials[i];
    sums[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t h = 512u; h > 0u; h >>= 1) {
        if (threadIdx.x < h) sums[threadIdx.x] += sums[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0u) *out = sums[0] / pixels;
}

}  // namespace dev

static dim3 flip_grid(uint32_t w, uint32_t h)
{
    return dim3((w + dev::kFlipTileX - 1) / dev::kFlipTileX, (h + dev::kFlipTileY - 1) / dev::kFlipTileY);
}

uint32_t flip_tiles(uint32_t w, uint32_t h)
{
    const dim3 g = flip_grid(w, h);
    return g.x * g.y;
}

hipError_t flip_error(const FlipArgs& a, double* mean, hipStream_t stream)
{
    const uint32_t n = a.w * a.h;
    hipLaunchKernelGGL(dev::flip_prepare_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid = flip_grid(a.w, a.h);
    // The tile and its seven x-filtered planes: 62 KB at the radius of the reference's viewing
    // geometry (10), 90 KB at the largest (16).
    const size_t rows = dev::kFlipTileY + 2 * a.r;
    const size_t lds = rows * ((dev::kFlipTileX + 2 * a.r) * sizeof(float4) + 7 * dev::kFlipTileX * sizeof(float));
    hipLaunchKernelGGL(dev::flip_error_kernel, grid, dim3(dev::kFlipThreads), (uint32_t)lds, stream, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(dev::flip_mean_kernel, dim3(1), dim3(1024), 0, stream, a.partials, grid.x * grid.y, (double)n,
                       mean);
    return hipGetLastError();
}

}  // namespace nbvh
