// generator.hip -- the small layers around the 3x3 convolutions of the
// MaterialGAN caller's StyleGAN2 synthesis network (src/materialgan.py:21-173,
// src/higan_models/stylegan2_generator_network.py:340-356,585-760), each as one
// kernel where a library call per layer costs more in launches than in work.
//
// Kernels
//   style_kernel          every layer's style, one matrix-vector product per
//                         layer, in one launch; style_grad_kernel and
//                         style_grad_sum_kernel: dL/dlatent.
//   torgb_kernel          the 1x1 convolution to the output channels with its
//                         style, plus the x2 upsampled skip image.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.hpp"
#include "../../include/svbrdf_hip.h"

using svbrdf_internal::check_launch;
using svbrdf_internal::fail;

namespace {

// ---------------------------------------------------------------------------
// Styles.  A wave takes one row of a layer at a time: 16-byte loads along the
// row, a butterfly sum.  The layers' tables travel as a kernel argument.  The
// 20 layers of the 256^2 generator (8,704 rows of 512, 18 MB) take 5.7 us; as
// a product per layer they took 20 launches of 7 us and as many bias copies.
constexpr int kMaxLayers = 32;
constexpr int kMaxDim = 4096;
constexpr int kRowsPerBlock = 16;    // forward: four waves of four rows
constexpr int kRowsPerSlice = 32;    // gradient: rows summed by one block

struct StyleTable {
    svbrdf_style_layer layer[kMaxLayers];
    int first[kMaxLayers + 1];       // first block of each layer
    int n;
};

// The layer of a block, and the block's index within it.
__device__ __forceinline__ int layer_of(const StyleTable &t, int block, int &local) {
    int l = 0;
    while (l + 1 < t.n && block >= t.first[l + 1]) ++l;
    local = block - t.first[l];
    return l;
}

__global__ __launch_bounds__(256) void style_kernel(StyleTable t, const float *__restrict__ latent, int dim,
                                                    float *__restrict__ out) {
    int local;
    const svbrdf_style_layer &y = t.layer[layer_of(t, blockIdx.x, local)];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float4 *v = reinterpret_cast<const float4 *>(latent + (size_t)y.row * dim);
#pragma unroll
    for (int k = 0; k < kRowsPerBlock / 4; ++k) {
        const int r = local * kRowsPerBlock + k * 4 + wave;
        if (r >= y.rows) break;
        const float4 *w = reinterpret_cast<const float4 *>(y.weight + (size_t)r * dim);
        float acc = 0.0f;
        for (int e = lane; e < dim / 4; e += 64) {
            const float4 a = w[e], b = v[e];
            acc += a.x * b.x;
            acc += a.y * b.y;
            acc += a.z * b.z;
            acc += a.w * b.w;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (lane == 0) out[y.offset + r] = acc * y.scale + y.bias[r] * y.bias_scale;
    }
}

// dL/dlatent: a block sums 32 rows of one layer, grad x weight, four columns
// per thread; then the slices of the layers that read a latent row are added
// in order.
__global__ __launch_bounds__(256) void style_grad_kernel(StyleTable t, const float *__restrict__ grad, int dim,
                                                         float *__restrict__ part) {
    int local;
    const svbrdf_style_layer &y = t.layer[layer_of(t, blockIdx.x, local)];
    const int r0 = local * kRowsPerSlice, r1 = min(y.rows, r0 + kRowsPerSlice);
    for (int e = threadIdx.x; e < dim / 4; e += 256) {
        const float4 *w = reinterpret_cast<const float4 *>(y.weight) + e;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
        for (int r = r0; r < r1; ++r) {
            const float4 a = w[(size_t)r * (dim / 4)];
            const float g = grad[y.offset + r];
            acc.x += g * a.x;
            acc.y += g * a.y;
            acc.z += g * a.z;
            acc.w += g * a.w;
        }
        acc.x *= y.scale; acc.y *= y.scale; acc.z *= y.scale; acc.w *= y.scale;
        reinterpret_cast<float4 *>(part + (size_t)blockIdx.x * dim)[e] = acc;
    }
}

__global__ __launch_bounds__(256) void style_grad_sum_kernel(StyleTable t, const float *__restrict__ part, int dim,
                                                             float *__restrict__ grad_latent) {
    const int e = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
    if (e >= dim) return;
    float acc = 0.0f;
    for (int l = 0; l < t.n; ++l) {
        if (t.layer[l].row != row) continue;
#pragma unroll 8
        for (int b = t.first[l]; b < t.first[l + 1]; ++b) acc += part[(size_t)b * dim + e];
    }
    grad_latent[(size_t)row * dim + e] = acc;
}

// ---------------------------------------------------------------------------
// y[o][p] = sum_c (weight[o][c] (style[c] scale)) x[c][p] (+ the skip image,
// upsampled as svbrdf_upsample2_blur).  The channels are split over a block's
// WAVES waves, VEC pixels per lane; the waves' sums meet in LDS.  Bound by
// latency on the small images (512 channels of 4^2 to 64^2: 6.8 to 7.4 us, with
// 8 waves and four loads in flight 8.0 to 8.7) and by reading x on the large
// ones: 128 channels of 256^2 (34 MB) take 10.5 us.  The library product, the
// scaling of its weights, the upsampling and the sum were 4 launches, 25 to 35 us.
constexpr int kMaxRgb = 9;
constexpr int kRgbPitch = 12;        // a channel's weights in LDS, three 16-byte reads

template <int VEC, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void torgb_kernel(const float *__restrict__ x, int cin, int h, int w,
                                                           const float *__restrict__ weight, int cout,
                                                           const float *__restrict__ style, float scale,
                                                           const float *__restrict__ skip, float *__restrict__ y) {
    typedef float vec __attribute__((ext_vector_type(VEC)));
    constexpr int PIXELS = 64 * VEC, AHEAD = 8;
    __shared__ float part[WAVES][kMaxRgb][PIXELS];
    extern __shared__ float4 wm4[];                       // [cin][kRgbPitch]
    float *wm = reinterpret_cast<float *>(wm4);
    const size_t HW = (size_t)h * w;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t p0 = (size_t)blockIdx.x * PIXELS, p = p0 + lane * VEC;
    const float *xp = x + (p < HW ? p : 0);               // HW is a multiple of VEC
    const int per = (cin + WAVES - 1) / WAVES;
    const int c0 = min(cin, wave * per), c1 = min(cin, c0 + per);
    const auto load = [&](int c) { return *reinterpret_cast<const vec *>(xp + (size_t)min(c, cin - 1) * HW); };
    vec v[AHEAD];                                         // in flight while the weights are scaled
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) v[k] = load(c0 + k);
    for (int c = threadIdx.x; c < cin; c += WAVES * 64) {
        const float s = style[c] * scale;
        float q[kMaxRgb];
#pragma unroll
        for (int o = 0; o < kMaxRgb; ++o) q[o] = weight[(size_t)min(o, cout - 1) * cin + c];
#pragma unroll
        for (int o = 0; o < kMaxRgb; ++o) wm[c * kRgbPitch + o] = q[o] * s;
    }
    __syncthreads();
    vec acc[kMaxRgb];
#pragma unroll
    for (int o = 0; o < kMaxRgb; ++o) acc[o] = 0.0f;
    for (int c = c0; c < c1; c += AHEAD) {
        vec u[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) u[k] = v[k];
        if (c + AHEAD < c1) {
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) v[k] = load(c + AHEAD + k);
        }
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            if (c + k >= c1) break;
            const float *m = wm + (c + k) * kRgbPitch;
#pragma unroll
            for (int o = 0; o < kMaxRgb; ++o) acc[o] += u[k] * m[o];
        }
    }
#pragma unroll
    for (int o = 0; o < kMaxRgb; ++o) *reinterpret_cast<vec *>(&part[wave][o][lane * VEC]) = acc[o];
    __syncthreads();
    for (int e = threadIdx.x; e < cout * PIXELS; e += WAVES * 64) {
        const int o = e / PIXELS, i = e - o * PIXELS;
        const size_t q = p0 + i;
        if (q >= HW) continue;
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) v += part[k][o][i];
        if (skip) {
            // out(2p) = (x(p-1) + 3 x(p)) / 4, out(2p+1) = (3 x(p) + x(p+1)) / 4 per axis
            const int hs = h / 2, ws = w / 2, oy = (int)(q / w), ox = (int)(q - (size_t)oy * w);
            const int ry = oy >> 1, rx = ox >> 1, ny = oy & 1 ? ry + 1 : ry - 1, nx = ox & 1 ? rx + 1 : rx - 1;
            const float *s = skip + (size_t)o * hs * ws;
            const bool my = ny >= 0 && ny < hs, mx = nx >= 0 && nx < ws;
            const float a = 0.75f * s[(size_t)ry * ws + rx] + (mx ? 0.25f * s[(size_t)ry * ws + nx] : 0.0f);
            const float b = my ? 0.75f * s[(size_t)ny * ws + rx] + (mx ? 0.25f * s[(size_t)ny * ws + nx] : 0.0f) : 0.0f;
            v += 0.75f * a + 0.25f * b;
        }
        y[(size_t)o * HW + q] = v;
    }
}

int check_layers(const char *what, const svbrdf_style_layer *layers, int n_layers, int dim, int rows, int latent_rows,
                 StyleTable &t) {
    if (n_layers < 1 || n_layers > kMaxLayers)
        return fail(SVBRDF_EINVAL, "%s: n_layers=%d outside [1, %d]", what, n_layers, kMaxLayers);
    if (dim < 4 || dim % 4 || dim > kMaxDim) return fail(SVBRDF_ESHAPE, "%s: dim=%d", what, dim);
    t.n = n_layers;
    t.first[0] = 0;
    for (int l = 0; l < n_layers; ++l) {
        const svbrdf_style_layer &y = layers[l];
        if (!y.weight || !y.bias) return fail(SVBRDF_EINVAL, "%s: null pointer in layer %d", what, l);
        if ((uintptr_t)y.weight & 15u) return fail(SVBRDF_EINVAL, "%s: layer %d is not 16-byte aligned", what, l);
        if (y.rows < 1 || y.rows > (1 << 20) || y.offset < 0 || y.row < 0 || y.row >= latent_rows)
            return fail(SVBRDF_ESHAPE, "%s: layer %d: rows=%d offset=%d row=%d", what, l, y.rows, y.offset, y.row);
        t.layer[l] = y;
        t.first[l + 1] = t.first[l] + (y.rows + rows - 1) / rows;
    }
    return SVBRDF_OK;
}

}  // namespace

extern "C" {

int svbrdf_style_layers(const svbrdf_style_layer *layers, int n_layers, const float *latent, int latent_rows, int dim,
                        float *styles, void *stream) {
    const char *what = "svbrdf_style_layers";
    if (!layers || !latent || !styles) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    if ((uintptr_t)latent & 15u) return fail(SVBRDF_EINVAL, "%s: latent must be 16-byte aligned", what);
    StyleTable t;
    if (int rc = check_layers(what, layers, n_layers, dim, kRowsPerBlock, latent_rows, t)) return rc;
    hipLaunchKernelGGL(style_kernel, dim3((unsigned)t.first[n_layers]), dim3(256), 0, (hipStream_t)stream, t, latent,
                       dim, styles);
    return check_launch(what);
}

size_t svbrdf_style_layers_grad_workspace_bytes(const svbrdf_style_layer *layers, int n_layers, int dim) {
    if (!layers || n_layers < 1 || n_layers > kMaxLayers || dim < 4 || dim > kMaxDim) return 0;
    size_t slices = 0;
    for (int l = 0; l < n_layers; ++l) slices += (size_t)(std::max(layers[l].rows, 0) + kRowsPerSlice - 1) / kRowsPerSlice;
    return slices * dim * sizeof(float);
}

int svbrdf_style_layers_grad(const svbrdf_style_layer *layers, int n_layers, const float *grad_styles, int latent_rows,
                             int dim, float *grad_latent, void *workspace, size_t workspace_bytes, void *stream) {
    const char *what = "svbrdf_style_layers_grad";
    if (!layers || !grad_styles || !grad_latent || !workspace)
        return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    if (latent_rows < 1 || latent_rows > 65535) return fail(SVBRDF_ESHAPE, "%s: latent_rows=%d", what, latent_rows);
    StyleTable t;
    if (int rc = check_layers(what, layers, n_layers, dim, kRowsPerSlice, latent_rows, t)) return rc;
    const size_t need = svbrdf_style_layers_grad_workspace_bytes(layers, n_layers, dim);
    if (workspace_bytes < need)
        return fail(SVBRDF_ESPACE, "%s: workspace of %zu bytes < %zu needed", what, workspace_bytes, need);
    if ((uintptr_t)workspace & 15u) return fail(SVBRDF_EINVAL, "%s: workspace must be 16-byte aligned", what);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(style_grad_kernel, dim3((unsigned)t.first[n_layers]), dim3(256), 0, s, t, grad_styles, dim,
                       (float *)workspace);
    if (int rc = check_launch(what)) return rc;
    hipLaunchKernelGGL(style_grad_sum_kernel, dim3((unsigned)(dim + 255) / 256, (unsigned)latent_rows), dim3(256), 0, s,
                       t, (const float *)workspace, dim, grad_latent);
    return check_launch(what);
}

int svbrdf_torgb(const float *x, int cin, int height, int width, const float *weight, int cout, const float *style,
                 float scale, const float *skip, float *y, void *stream) {
    const char *what = "svbrdf_torgb";
    if (!x || !weight || !style || !y) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    // 36 KB of weights beside the waves' sums
    if (cin < 1 || cin > 768 || cout < 1 || cout > kMaxRgb || height < 1 || width < 1 || height > 8192 || width > 8192)
        return fail(SVBRDF_ESHAPE, "%s: cin=%d cout=%d height=%d width=%d", what, cin, cout, height, width);
    if (skip && (height % 2 || width % 2))
        return fail(SVBRDF_ESHAPE, "%s: a skip image needs an even size, got %dx%d", what, height, width);
    const size_t HW = (size_t)height * width;
    const size_t lds = (size_t)cin * kRgbPitch * sizeof(float);
    hipStream_t s = (hipStream_t)stream;
    // Two pixels per lane and 8 waves where that still gives every compute unit
    // two blocks; on smaller images one and 16, so that fewer channels' loads
    // stand one behind the other.
    if (HW >= 2 * 256 * 128 && HW % 2 == 0 && ((uintptr_t)x & 7u) == 0)
        hipLaunchKernelGGL((torgb_kernel<2, 8>), dim3((unsigned)((HW + 127) / 128)), dim3(512), lds, s, x, cin, height,
                           width, weight, cout, style, scale, skip, y);
    else
        hipLaunchKernelGGL((torgb_kernel<1, 16>), dim3((unsigned)((HW + 63) / 64)), dim3(1024), lds, s, x, cin, height,
                           width, weight, cout, style, scale, skip, y);
    return check_launch(what);
}

}  // extern "C"
