// conv_common.hpp -- what the 3x3 convolution kernels of conv.hip and
// conv_split.hip share: the arguments, the epilogue, the K-split sum and the
// tiling helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "common.hpp"
#include "../../include/svbrdf_hip.h"

namespace svbrdf_internal {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kConvThreads = 256;   // four waves
constexpr int kMaxChannels = 4096;
constexpr int kMaxSide = 8192;
constexpr int kDirectMaxCout = 8;     // conv3x3_direct_kernel up to this many output channels
constexpr int kMaxSlices = 64;
constexpr int kComputeUnits = 256;    // MI355X

struct ConvArgs {
    const float *x;       // [N, Cin, H, W]
    const float *w;       // [9][Cin][Cout]
    const float *bias;    // [Cout] or null
    const float *noise;   // [H, W] or null
    float noise_strength;
    int act;              // SVBRDF_ACT_*
    // input gate: x is read as x * (gate > 0 ? gate_pos : gate_neg) where gate
    // is not null ([N, Cin, H, W], the forward output of the layer whose input
    // gradient this convolution computes: the activation's derivative)
    const float *gate;
    float gate_pos, gate_neg;
    float *y;             // [N, Cout, H, W]
    float *tap;           // a second copy of y, times tap_scale, or null
    float tap_scale;
    float *pool;          // the 2 x 2 averages of y [N, Cout, H / 2, W / 2], or null; y may then be null
    float *part;          // [slices][N, Cout, H, W] partial sums when K is split, else null
    int n, cin, cout, h, w_;
    int tw, th, tiles_x;  // pixel tile: th rows x tw columns
    int slices, cps;      // K slices (blockIdx.z = image x slices + slice) of cps chunks each
};

__device__ __forceinline__ float activate(float v, int act) {
    if (act == SVBRDF_ACT_RELU) return v > 0.0f ? v : 0.0f;
    if (act == SVBRDF_ACT_LRELU) return (v > 0.0f ? v : v * 0.2f) * 1.41421356237309515f;
    return v;
}

// the epilogue of output channel co at pixel p: noise, bias, activation
__device__ __forceinline__ float finish(const ConvArgs &a, float v, int co, size_t p) {
    if (a.noise) v = v + a.noise_strength * a.noise[p];
    if (a.bias) v = v + a.bias[co];
    return activate(v, a.act);
}

inline int pick_tile_width(int w) {
    int tw = 4;
    while (tw < w && tw < 32) tw *= 2;
    return tw;
}

inline bool conv_shape_ok(int n, int cin, int height, int width, int cout) {
    return n >= 1 && n <= 65535 && cin >= 1 && cout >= 1 && cin <= kMaxChannels && cout <= kMaxChannels &&
           height >= 1 && width >= 1 && height <= kMaxSide && width <= kMaxSide;
}

// Adds the K slices' partial sums a.part in slice order and applies the epilogue (conv.hip).
__attribute__((visibility("hidden"))) void launch_split_sum(const ConvArgs &a, hipStream_t s);

// Checks, plans and launches a convolution on the fp32 instruction (conv.hip).
__attribute__((visibility("hidden"))) int run_conv(const char *what, ConvArgs a, void *workspace,
                                                   size_t workspace_bytes, hipStream_t s);

// Estimated time (us, without its launch) of a convolution on the fp32
// instruction of more than kDirectMaxCout output and 4 input channels (conv.hip).
__attribute__((visibility("hidden"))) double conv_us(int n, int cin, int h, int w, int cout);

// Fills the epilogue-independent arguments of an input-gradient call (conv.hip).
__attribute__((visibility("hidden"))) ConvArgs input_grad_args(const float *grad_y, const float *y, int activation,
                                                               int n, int cout, int height, int width, int cin,
                                                               float *grad_x);

// The weight gradient on split operands (conv_split.hip): its tiling with the
// estimated time, and the launch; out: [slices][Cout][Cin][9].
struct WgradSplitPlan {
    int strips, n_chunks, co_tiles, ci_tiles, slices, cps;
    double us;
};
__attribute__((visibility("hidden"))) WgradSplitPlan plan_wgrad_split(int n, int cin, int h, int w, int cout);
__attribute__((visibility("hidden"))) void launch_wgrad_split(const WgradSplitPlan &p, const float *x,
                                                              const float *grad_z, int n, int cin, int h, int w,
                                                              int cout, float *out, hipStream_t s);

}  // namespace svbrdf_internal
