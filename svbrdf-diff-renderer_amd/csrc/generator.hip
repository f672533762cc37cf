// generator.hip -- the small layers around the 3x3 convolutions of the
// MaterialGAN caller's StyleGAN2 synthesis network (src/materialgan.py:21-173,
// src/higan_models/stylegan2_generator_network.py:340-356,585-760), each as one
// kernel where a library call per layer costs more in launches than in work.
//
// Kernels
//   style_kernel          every layer's style, one matrix-vector product per
//                         layer, in one launch; style_grad_kernel and
//                         style_grad_sum_kernel: dL/dlatent.
//   modconv_small_kernel  a modulated 3x3 convolution of at most 128 pixels
//                         straight from the network's weights, and
//                         modconv_small_sum_kernel: its K slices' sum with
//                         the demodulation and the epilogue.
//   torgb_kernel          the 1x1 convolution to the output channels with its
//                         style, plus the x2 upsampled skip image.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdint>

#include "conv_common.hpp"

using namespace svbrdf_internal;

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

// ---------------------------------------------------------------------------
// The modulated 3x3 convolution of the generator's first layers (4 x 4 and
// 8 x 8 pixels, 512 channels).  There the weights are the work: packing them
// with the style reads and writes all of them before the convolution reads
// them again.  Here a lane's weights go from the [Cout][Cin][3][3] layout
// straight to the MFMA's operand, 16 bytes along K = Cin x 9 at a time (lane
// half h takes the k = 8 q + 4 h + j of step (q, j)), times scale and style in
// the packing's order, and the squares for the demodulation factor are summed
// on the way; the factor multiplies the sums instead of the weights.  Input
// channels are staged in LDS with a one-pixel halo.  Up to 64 pixels the block's
// four waves split K and add up through LDS, above that they split the pixels.
// K is split over the blocks too; modconv_small_sum_kernel adds the slices.
// Bound by the latency of one or a few rounds (weights, staging, 36 steps).
// 512 -> 512, this path / packed: 4 x 4 10.8 / 29.0 us, 8 x 8 15.9 / 29.7, 11 x 11
// 24.7 / 36.0; 256 -> 256 at 4 x 4 9.7 / 17.9, 96 -> 96 at 8 x 8 13.9 / 13.8. Its
// redundant weight loads grow with the pixels and the packed path's do not: at
// 16 x 16 37.1 / 39.2 in a loop and no gain between other kernels, so it ends at
// 128. Prefetching the next round's weights or 512 blocks: no gain.
constexpr int kSmallMaxPixels = 128;
constexpr int kSmallUnit = 8;          // input channels of a wave's round: 72 products, 9 x 16 bytes
constexpr int kSmallBlocks = 256;

struct SmallArgs {
    const float *x, *w, *style;
    float scale;
    int cin, cout, h, w_, rounds, slices;   // rounds: per slice
    float *part, *squares;                  // [slices][Cout][H W], [slices][Cout]
};

template <int NT, bool SPLITK>
__global__ __launch_bounds__(256) void modconv_small_kernel(SmallArgs a) {
    constexpr int CI = SPLITK ? 4 * kSmallUnit : kSmallUnit;   // channels staged a round
    constexpr int HALO = SPLITK ? 3 * 66 : 3 * 130;            // the largest (h + 2) (w + 2)
    __shared__ float xs[CI * HALO];
    __shared__ float sq4[4][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, col = lane & 31, co0 = blockIdx.x * 32, slice = blockIdx.y;
    const int H = a.h, W = a.w_, P = H * W, w2 = W + 2, PH = (H + 2) * w2;
    const float *wrow = a.w + (size_t)min(co0 + col, a.cout - 1) * a.cin * 9;
    const int unit0 = SPLITK ? wave * kSmallUnit : 0;          // the wave's channels of a round
    int base[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int p = min(((SPLITK ? 0 : wave * NT) + n) * 32 + col, P - 1);
        base[n] = unit0 * PH + p / W * w2 + p % W;
    }
    v16f acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.0f;
    float sq = 0.0f;
    const int c_end = min((slice + 1) * a.rounds * CI, a.cin);
    for (int c0 = slice * a.rounds * CI; c0 < c_end; c0 += CI) {
        // Cin is a multiple of a unit: a wave's channels all exist or none does
        const int cu = c0 + unit0;
        const bool any = cu < a.cin;
        const float4 *wv = reinterpret_cast<const float4 *>(wrow + (size_t)(any ? cu : 0) * 9) + half;
        float4 v[9];
        float st[kSmallUnit];
#pragma unroll
        for (int q = 0; q < 9; ++q) v[q] = wv[2 * q];
#pragma unroll
        for (int c = 0; c < kSmallUnit; ++c) st[c] = a.style ? a.style[(any ? cu : 0) + c] : 1.0f;
        for (int e = tid; e < CI * PH; e += 256) {
            const int c = e / PH, q = e - c * PH, y = q / w2 - 1, x = q % w2 - 1;
            const bool in = c0 + c < a.cin && y >= 0 && y < H && x >= 0 && x < W;
            const float t = a.x[in ? (size_t)(c0 + c) * P + y * W + x : 0];
            xs[e] = in ? t : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const float wq[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k0 = 8 * q + j, k1 = k0 + 4, c0k = k0 / 9, t0 = k0 % 9, c1k = k1 / 9, t1 = k1 % 9;
                float m = wq[j] * a.scale * (half ? st[c1k] : st[c0k]);
                m = any ? m : 0.0f;
                sq += m * m;
                const int off = half ? c1k * PH + t1 / 3 * w2 + t1 % 3 : c0k * PH + t0 / 3 * w2 + t0 % 3;
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(m, xs[base[n] + off], acc[n], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    sq += __shfl_xor(sq, 32, 64);
    if constexpr (SPLITK) {
        if (half == 0) sq4[wave][col] = sq;
        if (wave > 0)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) xs[((wave - 1) * NT + n) * 1024 + r * 64 + lane] = acc[n][r];
        __syncthreads();
        if (wave > 0) return;
        sq = ((sq4[0][col] + sq4[1][col]) + sq4[2][col]) + sq4[3][col];
#pragma unroll
        for (int v = 0; v < 3; ++v)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] += xs[(v * NT + n) * 1024 + r * 64 + lane];
    }
    if (wave == 0 && half == 0 && co0 + col < a.cout) a.squares[(size_t)slice * a.cout + co0 + col] = sq;
    // element r of a tile: row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32
    float *out = a.part + (size_t)slice * a.cout * P;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int p = ((SPLITK ? 0 : wave * NT) + n) * 32 + col;
        if (p >= P) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int co = co0 + (r >> 2) * 8 + half * 4 + (r & 3);
            if (co < a.cout) out[(size_t)co * P + p] = acc[n][r];
        }
    }
}

// One output from the weights times the demodulation factor, as packed weights
// give it.  Where the factor is far from 1 the sums above, which it multiplies
// afterwards, can overflow or leave the normal range while the output does not;
// one thread's serial loop, for those alone.
__device__ float modulated_sum(const SmallArgs &a, int co, int p, float factor) {
    const int P = a.h * a.w_, y0 = p / a.w_, x0 = p - y0 * a.w_;
    float acc = 0.0f;
#pragma unroll 1
    for (int c = 0; c < a.cin; ++c) {
        const float s = a.style ? a.style[c] : 1.0f;
        const float *w = a.w + ((size_t)co * a.cin + c) * 9, *xc = a.x + (size_t)c * P;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int y = y0 + t / 3 - 1, x = x0 + t % 3 - 1;
            const bool in = y >= 0 && y < a.h && x >= 0 && x < a.w_;
            const float v = xc[in ? y * a.w_ + x : 0];
            acc += w[t] * a.scale * s * factor * (in ? v : 0.0f);
        }
    }
    return acc;
}

// c: the epilogue's arguments; c.part and squares as written above.
__global__ __launch_bounds__(256) void modconv_small_sum_kernel(ConvArgs c, SmallArgs a, int demodulate) {
    const float *__restrict__ squares = a.squares;
    const int P = c.h * c.w_, total = c.cout * P, e = blockIdx.x * 256 + threadIdx.x;
    if (e >= total) return;
    const int co = e / P;
    float v = 0.0f, sq = 0.0f;
    for (int s0 = 0; s0 < c.slices; s0 += 8) {   // eight loads of each in flight
        float pv[8], qv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int s = min(s0 + u, c.slices - 1);
            pv[u] = c.part[(size_t)s * total + e];
            qv[u] = squares[(size_t)s * c.cout + co];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (s0 + u < c.slices) {
                v += pv[u];
                sq += qv[u];
            }
        }
    }
    if (demodulate) {
        const float factor = rsqrtf(sq + 1e-8f), size = fabsf(v);
        const bool kept = size == 0.0f || (size >= 0x1p-100f && size <= FLT_MAX);
        v = kept ? v * factor : modulated_sum(a, co, e - co * P, factor);
    }
    c.y[e] = finish(c, v, co, e - co * P);
}

struct SmallPlan {
    bool taken;
    int co_tiles, rounds, slices;
};

SmallPlan plan_small(int cin, int h, int w, int cout) {
    SmallPlan p{};
    if (!conv_shape_ok(1, cin, h, w, cout) || (long long)h * w > kSmallMaxPixels || cin % kSmallUnit) return p;
    const int ci = h * w <= 64 ? 4 * kSmallUnit : kSmallUnit, total = (cin + ci - 1) / ci;
    p.taken = true;
    p.co_tiles = (cout + 31) / 32;
    const int want = std::max(1, std::min(total, kSmallBlocks / p.co_tiles));
    p.rounds = (total + want - 1) / want;
    p.slices = (total + p.rounds - 1) / p.rounds;
    return p;
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

size_t svbrdf_modconv3x3_small_workspace_bytes(int cin, int height, int width, int cout) {
    const SmallPlan p = plan_small(cin, height, width, cout);
    return p.taken ? (size_t)p.slices * cout * ((size_t)height * width + 1) * sizeof(float) : 0;
}

int svbrdf_modconv3x3_small(const float *x, int cin, int height, int width, const float *weight, int cout,
                            const float *style, float scale, int demodulate, const float *bias, const float *noise,
                            float noise_strength, int activation, float *y, void *workspace, size_t workspace_bytes,
                            void *stream) {
    const char *what = "svbrdf_modconv3x3_small";
    if (!x || !weight || !y || !workspace) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    const size_t need = svbrdf_modconv3x3_small_workspace_bytes(cin, height, width, cout);
    if (!need)
        return fail(SVBRDF_ESHAPE, "%s: cin=%d (a multiple of %d) cout=%d height=%d width=%d (at most %d pixels)", what,
                    cin, kSmallUnit, cout, height, width, kSmallMaxPixels);
    if (activation < SVBRDF_ACT_NONE || activation > SVBRDF_ACT_LRELU)
        return fail(SVBRDF_EINVAL, "%s: unknown activation %d", what, activation);
    if (workspace_bytes < need)
        return fail(SVBRDF_ESPACE, "%s: workspace of %zu bytes < %zu needed", what, workspace_bytes, need);
    if ((uintptr_t)weight & 15u) return fail(SVBRDF_EINVAL, "%s: weight must be 16-byte aligned", what);
    const SmallPlan p = plan_small(cin, height, width, cout);
    const int P = height * width;
    SmallArgs a{};
    a.x = x; a.w = weight; a.style = style; a.scale = scale; a.cin = cin; a.cout = cout; a.h = height; a.w_ = width;
    a.rounds = p.rounds; a.slices = p.slices;
    a.part = (float *)workspace;
    a.squares = a.part + (size_t)p.slices * cout * P;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)p.co_tiles, (unsigned)p.slices);
    if (P <= 32) hipLaunchKernelGGL((modconv_small_kernel<1, true>), grid, dim3(256), 0, s, a);
    else if (P <= 64) hipLaunchKernelGGL((modconv_small_kernel<2, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((modconv_small_kernel<1, false>), grid, dim3(256), 0, s, a);
    if (int rc = check_launch(what)) return rc;
    ConvArgs c{};
    c.bias = bias; c.noise = noise; c.noise_strength = noise_strength; c.act = activation;
    c.y = y; c.part = a.part; c.cout = cout; c.h = height; c.w_ = width; c.slices = p.slices;
    hipLaunchKernelGGL(modconv_small_sum_kernel, dim3((unsigned)((cout * P + 255) / 256)), dim3(256), 0, s, c, a,
                       demodulate);
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
