// conv_split.hip -- the 3x3 convolution of conv.hip (stride 1, zero padding
// 1, the same epilogues and input gate) at fp32 precision on the bf16 matrix
// cores.
//
// v_mfma_f32_32x32x2f32 runs at 135 TFLOP/s on an MI355X, v_mfma_f32_32x32x16_bf16
// at 1,970 (both measured from registers).  An fp32 value is the sum of three
// bf16 values, x = h + m + l: each is the rounding of what the ones before
// leave, 8 significant bits apiece, 24 in all.  A product is then
//   x w = hh' + (hm' + mh') + (hl' + mm' + lh') + O(2^-25 |x w|),
// six bf16 products that the matrix core multiplies exactly and accumulates
// in fp32, at 1,970 / 6 = 328 TFLOP/s.  bf16 has fp32's exponent, so nothing is
// scaled; what lies at either end of the range is taken apart (below).
//
// Precision.  The hh' products and the five small ones have accumulators of
// their own, so the sum is rounded at its own size once per 16 products (the
// fp32 instruction: once per product pair).  The bf16 instruction drops what
// it shifts out of its adder towards minus infinity, a bias that the adjoint
// of an upsampling adds up coherently; so the weights of every odd chunk are
// negated and the accumulators with them, and the bias of one chunk cancels
// the next one's.  Relative error against 64 bits (fp32 instruction / this;
// normal values, 3 x 3 taps): 64 channels 2.9e-7 / 1.6e-7, 128: 6.1e-7 /
// 2.0e-7, 256: 8.6e-7 / 2.9e-7, 512 at 64^2: 6.0e-7 (in K slices) / 2.9e-7;
// with log-normal magnitudes (sigma 3) 5.7e-7 / 2.3e-7.  The mean error is
// below 2e-10 of sum |x w|.  With one accumulator per sum and no sign
// change it was 5.2e-7 at 128 channels with a mean of -3e-9, and the W+
// gradient through the 13 layers of the generator was 3.1e-5 off; it is
// 1.0e-6, and 1.4e-6 on the fp32 instruction.
//
// Values that do not split: infinities and NaN, finite values that round to
// infinity in bf16 (above 3.39e38), and small ones (2^-102) whose last term
// would leave bf16's normal range (exact down to 2^-110, 8 bits short at
// 2^-118, lost at 2^-133).  Such an operand puts a NaN among its tile's, and a
// wave whose sums come out NaN, infinite or themselves below 2^-100 repeats
// its tile from the fp32 values on the fp32 instruction (redo_fp32), so they
// count and spread exactly as in conv.hip.  The check costs 0.2 to 0.3 % of a
// convolution and 1 % of a modulated layer's pass; one such pixel in 9 x 64 ->
// 64 at 256^2 nothing to be seen, all of them 1,750 us (fp32 kernel 390-450).
//
// Kernels
//   split_factor_kernel   the demodulation factor of each output channel.
//   split_pack_kernel     weights -> the matrix core's operand order, split:
//                         [K chunk of 16][tap][h, m, l][32 outputs][lane][8].
//   conv3x3_split_kernel  the convolution.
//   conv3x3_wgrad_split_kernel
//                         its weight gradient.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "conv_common.hpp"

using namespace svbrdf_internal;

namespace {

constexpr int kThreads = kConvThreads;
constexpr int kKC = 16;   // input channels per chunk: one MFMA's K

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

__host__ __device__ constexpr int chunks_of(int k) { return (k + kKC - 1) / kKC; }
// The first of a chunk's 16 channels.  The last chunk of a K that is no
// multiple of 16 reaches back: its weights for the channels of the chunk
// before are zero, so every chunk reads 16 channels that exist.
__host__ __device__ constexpr int chunk_base(int chunk, int k) { return chunk * kKC + kKC <= k ? chunk * kKC : k - kKC; }
// groups of 32 output channels; even, so that a wave's 64 channels exist
__host__ __device__ constexpr int groups_of(int m) { return (m + 63) / 64 * 2; }

__device__ __forceinline__ float bf_lo(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf_hi(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

// h + m + l of two finite values, as packed bf16 pairs.  No contraction: the
// value is the rounded product that a caller passes, not the product itself.
// True where a last term leaves bf16's normal range, so that it may be off: the
// rest is a subnormal number there (a compare per value; 0 and every value of
// 2^-102 or more have none).
__device__ __forceinline__ bool split_pair(float a, float b, unsigned &h, unsigned &m, unsigned &l) {
#pragma clang fp contract(off)
    h = __builtin_bit_cast(unsigned, v2bf{(__bf16)a, (__bf16)b});
    a -= bf_lo(h);
    b -= bf_hi(h);
    m = __builtin_bit_cast(unsigned, v2bf{(__bf16)a, (__bf16)b});
    a -= bf_lo(m);
    b -= bf_hi(m);
    l = __builtin_bit_cast(unsigned, v2bf{(__bf16)a, (__bf16)b});
    constexpr int kSubnormal = 0x90;
    return __builtin_amdgcn_classf(a, kSubnormal) | __builtin_amdgcn_classf(b, kSubnormal);
}

// ---------------------------------------------------------------------------
// Weights.  The factor of an output channel is the one of conv.hip's packing:
// the same per-thread order, so the same bits.
__global__ __launch_bounds__(kThreads) void split_factor_kernel(const float *__restrict__ w, int cin,
                                                                const float *__restrict__ style, float scale,
                                                                float *__restrict__ factor) {
    __shared__ float red[kThreads / 64];
    const int n = cin * 9;
    const float *wc = w + (size_t)blockIdx.x * n;
    float acc = 0.0f;
    // six elements' loads in flight (512 rows of 512 channels: 8.1 -> 4.7 us)
    constexpr int U = 6;
    int e = threadIdx.x;
    for (; e + (U - 1) * kThreads < n; e += U * kThreads) {
        float v[U], sv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            v[u] = wc[e + u * kThreads];
            sv[u] = style ? style[(e + u * kThreads) / 9] : 1.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float x = v[u] * scale * sv[u];
            acc += x * x;
        }
    }
    for (; e < n; e += kThreads) {
        const float v = wc[e] * scale * (style ? style[e / 9] : 1.0f);
        acc += v * v;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) factor[blockIdx.x] = rsqrtf(((red[0] + red[1]) + red[2]) + red[3] + 1e-8f);
}

// Non-zero values below 2^-100 do not split: (bits << 1) - 1 orders magnitudes
// as unsigned numbers, with zero above all.
constexpr unsigned kTiny = (27u << 24) - 1u;
__device__ __forceinline__ unsigned rank_of(float v) { return (__float_as_uint(v) << 1) - 1u; }
// A NaN in both halves of a packed pair.  As a weight's first term it marks a
// value that does not split: its other two then hold the fp32 bits.
constexpr unsigned kMark = 0x7fffu, kMarkPair = 0x7fff7fffu;

enum PackForm {
    kNatural,      // [M, K, 3, 3]
    kTransposed,   // [K, M, 3, 3], taps flipped: the input gradient's weights
    kPacked,       // [9][K][M]: svbrdf_conv3x3_pack's output
};

// One block per 32 outputs and 16-channel chunk: the source rows go to LDS as
// they lie in memory (runs of 144, 288 or 32 floats), then each thread writes
// the 16 bytes of a lane's operand for one tap and term: 1 KB per wave and
// store, contiguous.  A bandwidth-bound pass over 10 bytes per weight: 512 x
// 512 (24 MB) in 7.0 us from the layer's weights, 9.6 from packed ones (12.4
// and 14.0 with the loads one behind the other).
template <PackForm FORM>
__global__ __launch_bounds__(kThreads) void split_pack_kernel(const float *__restrict__ w, int m_total, int k_total,
                                                              const float *__restrict__ style, float scale,
                                                              const float *__restrict__ factor,
                                                              uint4 *__restrict__ out) {
    constexpr int ROWS = FORM == kNatural ? 32 : FORM == kTransposed ? kKC : 9 * kKC;
    constexpr int RUN = FORM == kNatural ? kKC * 9 : FORM == kTransposed ? 32 * 9 : 32;
    constexpr int PITCH = RUN + 1;
    constexpr int PER = ROWS * RUN / kThreads;   // 18, whichever the form
    static_assert(ROWS * RUN == PER * kThreads, "whole passes");
    __shared__ float tile[ROWS * PITCH];
    __shared__ float by_m[32], by_k[kKC];        // a weight's factors by output and by input channel
    const int groups = groups_of(m_total);
    const int m0 = blockIdx.x * 32, chunk = blockIdx.y;
    const int k0 = chunk_base(chunk, k_total), skip = chunk * kKC - k0;   // channels of the chunk before
    float v[PER];   // all loads in flight: a valid address and a select
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = threadIdx.x + i * kThreads;
        const int r = e / RUN, c = e - r * RUN;
        bool ok;
        size_t o;
        if constexpr (FORM == kNatural) {
            ok = m0 + r < m_total && c / 9 >= skip;
            o = ((size_t)(m0 + r) * k_total + k0) * 9 + c;
        } else if constexpr (FORM == kTransposed) {
            ok = r >= skip && m0 + c / 9 < m_total;
            o = ((size_t)(k0 + r) * m_total + m0) * 9 + c;
        } else {
            const int t = r / kKC, k = r % kKC;
            ok = k >= skip && m0 + c < m_total;
            o = ((size_t)t * k_total + k0 + k) * m_total + m0 + c;
        }
        const float x = w[ok ? o : 0];
        v[i] = ok ? x : 0.0f;
    }
    if constexpr (FORM != kPacked) {
        // the style belongs to the layer's input channels, the demodulation
        // factor to its output channels
        if (threadIdx.x < 32) {
            const int m = min(m0 + (int)threadIdx.x, m_total - 1);
            const float *f = FORM == kNatural ? factor : style;
            by_m[threadIdx.x] = f ? f[m] : 1.0f;
        } else if (threadIdx.x < 32 + kKC) {
            const float *f = FORM == kNatural ? style : factor;
            by_k[threadIdx.x - 32] = f ? f[k0 + threadIdx.x - 32] : 1.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = threadIdx.x + i * kThreads;
        const int r = e / RUN, c = e - r * RUN;
        tile[r * PITCH + c] = v[i];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < 9 * 64; q += kThreads) {
        const int t = q / 64, lane = q & 63;
        const int mm = lane & 31, kk = (lane >> 5) * 8;
        uint4 term[3];
        unsigned *h = &term[0].x, *md = &term[1].x, *l = &term[2].x;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            float v[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int k = kk + j + i;
                if constexpr (FORM == kPacked) v[i] = tile[(t * kKC + k) * PITCH + mm];
                else if constexpr (FORM == kNatural) v[i] = tile[mm * PITCH + k * 9 + t] * scale * by_k[k] * by_m[mm];
                else v[i] = tile[k * PITCH + mm * 9 + (8 - t)] * scale * by_m[mm] * by_k[k];
                v[i] = chunk & 1 ? -v[i] : v[i];
            }
            const bool tiny = split_pair(v[0], v[1], h[j / 2], md[j / 2], l[j / 2]);
            const bool huge = (h[j / 2] & 0x7f80u) == 0x7f80u || (h[j / 2] & 0x7f800000u) == 0x7f800000u;
            if (tiny || huge) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const unsigned sh = i * 16, keep = 0xffff0000u >> sh, bits = __float_as_uint(v[i]);
                    if (((h[j / 2] >> sh) & 0x7f80u) != 0x7f80u && rank_of(v[i]) >= kTiny) continue;
                    h[j / 2] = (h[j / 2] & keep) | (kMark << sh);
                    md[j / 2] = (md[j / 2] & keep) | (bits >> 16 << sh);
                    l[j / 2] = (l[j / 2] & keep) | ((bits & 0xffffu) << sh);
                }
            }
        }
#pragma unroll
        for (int s = 0; s < 3; ++s)
            out[(((size_t)(chunk * 9 + t) * 3 + s) * groups + blockIdx.x) * 64 + lane] = term[s];
    }
}

// ---------------------------------------------------------------------------
// The convolution.  Block tile 64 WM output channels x 64 WN pixels (th rows x
// tw columns), four waves of 64 x 64 (2 x 2 MFMA tiles of 32 x 32).  Per chunk
// of 16 input channels the block splits its input tile with a one-pixel halo
// into LDS, in the operand's order: plane (term, half of the 16 channels),
// then pixel, 16 bytes each, so a lane's operand for a tap is one aligned
// ds_read_b128 and the lanes of a half-wave read consecutive ones.  The
// weights come straight from global memory, already in operand order (1 KB
// per wave and load, L1 / L2 hits: the blocks of an output group walk the
// same chunks), one tap ahead of their use.  The next chunk's input loads are
// issued before this chunk's 9 x 24 MFMAs and split into the other LDS buffer
// beside the last taps' MFMAs, so a block has one short barrier per chunk.
//
// Bound by the matrix cores, and those by power: 55 to 65 % busy at 1.96 to 2.05
// GHz (peak 2.4), where all-register MFMAs reach 1.88.  9 x 64 -> 64 at 256^2
// with inputs behind a ReLU: 230 us = 189 TFLOP/s of fp32 products (fp32
// instruction 387 us), 256 -> 128 at 256^2: 172 us, 224 TFLOP/s (333 us); inputs
// without zeros draw more power, 265-300 us for the first.  Splitting after the MFMAs instead of beside
// them: 249 and 189 us; weights loaded where they are used: 310 and 234 us.
// Three waves per SIMD (168 registers) gain nothing: 227 and 179 us.
constexpr int halo_pixels(int wn) { return wn == 4 ? 340 : 204; }   // largest (th + 2)(tw + 2), see plan

struct SplitArgs {
    ConvArgs c;
    const uint4 *w;   // split_pack_kernel's output
};

// The fp32 value of a split weight: output m, input channel k, tap t.
__device__ __forceinline__ float split_weight(const uint4 *w, int groups, int k_total, int m, int k, int t) {
    const int chunk = k / kKC, kk = k - chunk_base(chunk, k_total);
    const size_t base = ((size_t)(chunk * 9 + t) * 3 * groups + m / 32) * 64 + (m & 31) + 32 * (kk >> 3);
    const size_t step = (size_t)groups * 64;
    unsigned v[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) v[s] = reinterpret_cast<const unsigned short *>(w + base + s * step)[kk & 7];
    const float x = v[0] == kMark ? __uint_as_float(v[1] << 16 | v[2])
                                  : bf_lo(v[0]) + (bf_lo(v[1]) + bf_lo(v[2]));
    return chunk & 1 ? -x : x;
}

// Element r of MFMA tile (i, j): row 8 (r / 4) + 4 (lane / 32) + r % 4, column
// lane % 32.  ACT: the activation, or kPartial for a K slice's raw sums.
constexpr int kPartial = -1;
template <int ACT, bool TAP = false>
__device__ __forceinline__ void store_rows(const ConvArgs &a, float *out, int com, const int (&oy)[2],
                                           const int (&ox)[2], const v16f (&acc)[2][2]) {
    const int half = ((threadIdx.x >> 5) & 1) * 4;
    const size_t HW = (size_t)a.h * a.w_;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (oy[j] >= a.h || ox[j] >= a.w_) continue;
        const unsigned p = (unsigned)(oy[j] * a.w_ + ox[j]);
        // the lane's byte offset from a row's first pixel, at most 5 planes
        const unsigned off = (p + (unsigned)half * (unsigned)HW) * 4u;
        float nz = 0.0f;
        if (ACT != kPartial && a.noise) nz = a.noise_strength * a.noise[p];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = com + i * 32 + (r >> 2) * 8 + (r & 3);
                if (row + half >= a.cout) continue;
                float v = acc[i][j][r];
                if constexpr (ACT != kPartial) {
                    v = v + nz;
                    if (a.bias) v = v + a.bias[row + half];
                    v = activate(v, ACT);
                    if (TAP) v = v * a.tap_scale;
                }
                *reinterpret_cast<float *>(reinterpret_cast<char *>(out + (size_t)row * HW) + off) = v;
            }
    }
}

// The 2 x 2 averages of a tile of 32 columns: its two MFMA columns are two rows
// of the image, its even and odd lanes two columns.  Even lanes write, in
// avgpool2_kernel's order of operations.
template <int ACT>
__device__ __forceinline__ void store_pooled(const ConvArgs &a, int img, int com, const int (&oy)[2],
                                             const int (&ox)[2], const v16f (&acc)[2][2]) {
    const int half = ((threadIdx.x >> 5) & 1) * 4, hp = a.h / 2, wp = a.w_ / 2;
    const bool whole = !(threadIdx.x & 1) && oy[1] < a.h && ox[0] + 1 < a.w_;
    const size_t HP = (size_t)hp * wp;
    float *out = a.pool + (size_t)img * a.cout * HP;
    const unsigned off = ((unsigned)(oy[0] / 2 * wp + ox[0] / 2) + (unsigned)half * (unsigned)HP) * 4u;
    float nz[2] = {0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 2; ++j)
        if (a.noise && oy[j] < a.h && ox[j] < a.w_) nz[j] = a.noise_strength * a.noise[oy[j] * a.w_ + ox[j]];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = com + i * 32 + (r >> 2) * 8 + (r & 3);
            const float b = a.bias && row + half < a.cout ? a.bias[row + half] : 0.0f;
            float v[2], u[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                v[j] = acc[i][j][r] + nz[j];
                v[j] = activate(v[j] + b, ACT);
                u[j] = __shfl_xor(v[j], 1, 64);
            }
            if (!whole || row + half >= a.cout) continue;
            *reinterpret_cast<float *>(reinterpret_cast<char *>(out + (size_t)row * HP) + off) =
                (((v[0] + u[0]) + v[1]) + u[1]) / 4.0f;
        }
}

template <int ACT>
__device__ __forceinline__ void store_outputs(const ConvArgs &a, int img, int com, const int (&oy)[2],
                                              const int (&ox)[2], const v16f (&acc)[2][2]) {
    const size_t first = (size_t)img * a.cout * a.h * a.w_;
    if (a.y) store_rows<ACT>(a, a.y + first, com, oy, ox, acc);
    if (a.tap) store_rows<ACT, true>(a, a.tap + first, com, oy, ox, acc);
    if (a.pool) store_pooled<ACT>(a, img, com, oy, ox, acc);
}

__device__ __forceinline__ void store_tile(const ConvArgs &a, int img, int slice, int com, const int (&oy)[2],
                                           const int (&ox)[2], const v16f (&acc)[2][2]) {
    const size_t image = (size_t)a.cout * a.h * a.w_;
    if (a.part) store_rows<kPartial>(a, a.part + ((size_t)slice * a.n + img) * image, com, oy, ox, acc);
    else if (a.act == SVBRDF_ACT_RELU) store_outputs<SVBRDF_ACT_RELU>(a, img, com, oy, ox, acc);
    else if (a.act == SVBRDF_ACT_LRELU) store_outputs<SVBRDF_ACT_LRELU>(a, img, com, oy, ox, acc);
    else store_outputs<SVBRDF_ACT_NONE>(a, img, com, oy, ox, acc);
}

// A wave's 64 x 64 tile again on the fp32 instruction, from the fp32 inputs:
// only where the split sums were not finite.
__device__ __forceinline__ void redo_fp32(const SplitArgs &s, int img, int slice, int com, const int (&oy)[2],
                                          const int (&ox)[2], v16f (&acc)[2][2]) {
    const ConvArgs &a = s.c;
    const int lane = threadIdx.x & 63, groups = groups_of(a.cout);
    const size_t HW = (size_t)a.h * a.w_;
    const float *xi = a.x + (size_t)img * a.cin * HW;
    const float *gi = a.gate ? a.gate + (size_t)img * a.cin * HW : nullptr;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const int k_end = min((slice + 1) * a.cps * kKC, a.cin);
#pragma unroll 1
    for (int k0 = slice * a.cps * kKC; k0 < k_end; k0 += 2) {
        const int k = k0 + (lane >> 5);
#pragma unroll 1
        for (int t = 0; t < 9; ++t) {
            float av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int m = com + i * 32 + (lane & 31);
                av[i] = k < k_end && m < a.cout ? split_weight(s.w, groups, a.cin, m, k, t) : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int y = oy[j] + t / 3 - 1, x = ox[j] + t % 3 - 1;
                bv[j] = 0.0f;
                if (k < k_end && y >= 0 && y < a.h && x >= 0 && x < a.w_) {
                    const size_t o = (size_t)k * HW + (size_t)y * a.w_ + x;
                    bv[j] = gi ? xi[o] * (gi[o] > 0.0f ? a.gate_pos : a.gate_neg) : xi[o];
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
    }
}

template <int WM, int WN, bool GATE>
__global__ __launch_bounds__(kThreads, 2) void conv3x3_split_kernel(SplitArgs s) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int HALO = halo_pixels(WN);
    constexpr int PER = (2 * HALO + kThreads - 1) / kThreads;   // (pixel, channel octet) items per thread
    __shared__ uint4 tile[2][3][2 * HALO + 1];   // and a slot that items past the last write to
    const ConvArgs &a = s.c;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave - wm * WN;
    const int img = blockIdx.z / a.slices, slice = blockIdx.z - img * a.slices;
    const int groups = groups_of(a.cout);
    const int com = (blockIdx.y * WM + wm) * 64;                 // the wave's first output channel
    const int group = min(com / 32, groups - 2);                 // past the end: valid weights, nothing stored
    const int tyi = blockIdx.x / a.tiles_x, txi = blockIdx.x - tyi * a.tiles_x;
    const int y0 = tyi * a.th, x0 = txi * a.tw;
    const int tw2 = a.tw + 2, hs = (a.th + 2) * tw2;
    const int H = a.h, W = a.w_, HW = H * W;
    const size_t img_base = (size_t)img * a.cin * HW;

    // This thread's staging items: the byte offset of its pixel in its octet's
    // first plane (0 and !in: outside the image, read and not used), and where
    // it goes.  32 bits reach all of a chunk: 16 planes of at most 2^28 bytes.
    unsigned off[PER];
    int dst[PER];
    bool in[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int q = tid + k * kThreads;
        const int o = q >= hs ? 1 : 0, p = q - o * hs;
        const int r = p / tw2, c = p - r * tw2;
        const int yy = y0 - 1 + r, xx = x0 - 1 + c;
        in[k] = q < 2 * hs && yy >= 0 && yy < H && xx >= 0 && xx < W;
        off[k] = in[k] ? (o * 8u * (unsigned)HW + (unsigned)(yy * W + xx)) * 4u : 0u;
        dst[k] = q < 2 * hs ? o * HALO + p : 2 * HALO;
    }
    float xr[PER][8];
    unsigned open[PER];   // bit j: the gate of channel j is positive
    auto load_chunk = [&](const float *src, int chunk) {
        const char *xc = reinterpret_cast<const char *>(src + img_base + (size_t)chunk_base(chunk, a.cin) * HW);
#pragma unroll
        for (int k = 0; k < PER; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                xr[k][j] = *reinterpret_cast<const float *>(xc + (size_t)j * HW * 4 + off[k]);
    };
    // the gate passes through the same registers, a bit per value of it stays
    auto take_gate = [&]() {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            open[k] = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) open[k] |= xr[k][j] > 0.0f ? 1u << j : 0u;
        }
    };
    auto store_item = [&](int k, int buf) {
        uint4 t[3];
        unsigned *h = &t[0].x, *m = &t[1].x, *l = &t[2].x;
        bool tiny = false;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            float v[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                v[i] = xr[k][j + i];
                if constexpr (GATE) v[i] = v[i] * (open[k] >> (j + i) & 1 ? a.gate_pos : a.gate_neg);
                v[i] = in[k] ? v[i] : 0.0f;
            }
            tiny |= split_pair(v[0], v[1], h[j / 2], m[j / 2], l[j / 2]);
        }
        t[0].x = tiny ? kMarkPair : t[0].x;
#pragma unroll
        for (int i = 0; i < 3; ++i) tile[buf][i][dst[k]] = t[i];
    };

    // the halo-tile pixel each lane feeds to the two MFMA columns of its wave
    int pix[2], oy[2], ox[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int nn = wn * 64 + j * 32 + (lane & 31);
        const int ty = nn / a.tw, tx = nn - ty * a.tw;
        pix[j] = ty * tw2 + tx + (lane >> 5) * HALO;
        oy[j] = y0 + ty;
        ox[j] = x0 + tx;
    }
    // the h h' products and the five small ones, added at the end: one rounding
    // at the sum's own size per 16 products
    v16f acc[2][2], low[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.0f;

    const int n_chunks = chunks_of(a.cin);
    const int c_begin = slice * a.cps, c_end = min(n_chunks, c_begin + a.cps);
    const size_t term_step = (size_t)groups * 64, tap_step = 3 * term_step;
    // the weights of the next tap to load; the scheduling barriers keep the
    // loads a whole tap (768 matrix-core cycles) ahead of their use
    const uint4 *wp = s.w + (size_t)group * 64 + (size_t)c_begin * 9 * tap_step;
    const uint4 *const w_last = s.w + (size_t)group * 64 + ((size_t)c_end * 9 - 1) * tap_step;
    v8bf wreg[2][2][3];   // [buffer][MFMA row][term]
    auto load_weights = [&](int b) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) wreg[b][i][k] = __builtin_bit_cast(v8bf, (wp + k * term_step + i * 64)[lane]);
        wp = wp < w_last ? wp + tap_step : w_last;
    };
    if constexpr (GATE) {
        load_chunk(a.gate, c_begin);
        take_gate();
    }
    load_chunk(a.x, c_begin);
    load_weights(0);
#pragma unroll
    for (int k = 0; k < PER; ++k) store_item(k, 0);
    __syncthreads();
    auto run_chunk = [&](int c, auto last) {
        constexpr bool LAST = decltype(last)::value;
        const int buf = (c - c_begin) & 1;
        const uint4 *T = &tile[buf][0][0];
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            load_weights((t + 1) & 1);
            if constexpr (!LAST) {
                if (t == 0) load_chunk(GATE ? a.gate : a.x, c + 1);
                if (GATE && t == 3) {
                    take_gate();
                    load_chunk(a.x, c + 1);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            v8bf xv[2][3];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint4 *p = T + pix[j] + (t / 3) * tw2 + t % 3;
#pragma unroll
                for (int k = 0; k < 3; ++k) xv[j][k] = __builtin_bit_cast(v8bf, p[k * (2 * HALO + 1)]);
            }
            constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        v16f &d = q < 5 ? low[i][j] : acc[i][j];
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wreg[t & 1][i][TA[q]], xv[j][TB[q]], d, 0, 0, 0);
                    }
            // the next chunk's items are split beside the last taps' MFMAs
            if (!LAST && t + PER >= 9) store_item(t + PER - 9, buf ^ 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!LAST) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[i][j][r] = -acc[i][j][r];
                        low[i][j][r] = -low[i][j][r];
                    }
            // nine taps: the next chunk's first weights are in the odd buffer
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int k = 0; k < 3; ++k) wreg[0][i][k] = wreg[1][i][k];
            __syncthreads();
        }
    };
    for (int c = c_begin; c + 1 < c_end; ++c) run_chunk(c, std::false_type{});
    run_chunk(c_end - 1, std::true_type{});

    bool bad = false;
    unsigned least = ~0u;   // a sum below 2^-100 has low products that leave fp32's range
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] += low[i][j][r];
                acc[i][j][r] = c_end & 1 ? acc[i][j][r] : -acc[i][j][r];
                bad |= !(fabsf(acc[i][j][r]) <= FLT_MAX);
                least = min(least, rank_of(acc[i][j][r]));
            }
    if (__any(bad || least < kTiny)) redo_fp32(s, img, slice, com, oy, ox, acc);
    store_tile(a, img, slice, com, oy, ox, acc);
}

// ---------------------------------------------------------------------------
// The weight gradient (conv.hip's conv3x3_wgrad_kernel) on split operands: per
// tap a GEMM over the pixels, M = output channels, N = input channels.  A block
// of twelve waves owns 64 x 64 (co, ci) for all nine taps: a wave 32 x 32 of
// the three taps of one kernel row.  K runs over chunks of 32 pixels of one
// image row, down a strip of the image: the chunk's dL/dz and the input row
// below it go to LDS split, [term][row][pixel octet][channel] with 16 bytes of
// eight pixels each, so a lane's operand is one ds_read_b128; the input rows
// stay for the three chunks that read them (a ring of four).  The taps to the
// left and right are an octet shifted by a pixel in registers (v_alignbit) with
// the neighbouring octets' edge.  One block a compute unit: three waves per
// matrix core hide each other's reads, shifts and splits.  The sums and dL/dz
// change sign every second chunk, for the reason given above.
// The sums leave through LDS: a lane's are 9 floats apart in the output.
//
// Matrix cores 43 to 46 % busy at 2.2 GHz; what is left is the operand reads behind
// each chunk's barrier.  512 x 512 at 64^2: 122 us with the sum of 4 slices (159
// TFLOP/s; the fp32 kernel 223), 256 -> 128 at 256^2 222 (408).  Re-reading all
// three input rows for every chunk took 155 and 265, stores straight from the
// accumulators 8 to 14 more.  Error against 64 bits: 9.0e-8 (fp32 1.8e-7) for
// 128 x 128 at 64^2.
constexpr int kWgThreads = 768;
constexpr int kWgTile = 64;                      // output and input channels of a block
constexpr int kWgPixels = 32;                    // pixels of a chunk
constexpr int kWgOctets = kWgPixels / 8;
// An octet's 64 channels, plus 32 bytes: the stores of neighbouring octets
// meet different banks.
constexpr int kWgStride = kWgTile + 2;           // in 16-byte units

struct WgradSplitArgs {
    const float *x, *gz;
    float *out;
    int n, cin, cout, h, w_;
    int strips, n_chunks, cps;
};

__device__ __forceinline__ uint4 shifted_left(const uint4 &v, unsigned before) {   // pixels p - 1
    return make_uint4(__builtin_amdgcn_alignbit(v.x, before, 16), __builtin_amdgcn_alignbit(v.y, v.x, 16),
                      __builtin_amdgcn_alignbit(v.z, v.y, 16), __builtin_amdgcn_alignbit(v.w, v.z, 16));
}
__device__ __forceinline__ uint4 shifted_right(const uint4 &v, unsigned after) {   // pixels p + 1
    return make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, 16), __builtin_amdgcn_alignbit(v.z, v.y, 16),
                      __builtin_amdgcn_alignbit(v.w, v.z, 16), __builtin_amdgcn_alignbit(after, v.w, 16));
}

// A wave's sums again on the fp32 instruction: only where they were not finite.
__device__ __forceinline__ void redo_wgrad_fp32(const WgradSplitArgs &a, int c_begin, int c_end, int co, int ci, int dy,
                                                v16f (&acc)[3]) {
    const int lane = threadIdx.x & 63;
    const size_t HW = (size_t)a.h * a.w_;
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
#pragma unroll 1
    for (int c = c_begin; c < c_end; ++c) {
        const int y = c % a.h, strip = c / a.h % a.strips, img = c / a.h / a.strips;
        const int yy = y + dy - 1;
#pragma unroll 1
        for (int k = 0; k < kWgPixels; k += 2) {
            const int x = strip * kWgPixels + k + (lane >> 5);
            float g = 0.0f;
            if (co < a.cout && x < a.w_) g = a.gz[((size_t)img * a.cout + co) * HW + (size_t)y * a.w_ + x];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const int xx = x + t - 1;
                float v = 0.0f;
                if (ci < a.cin && yy >= 0 && yy < a.h && xx >= 0 && xx < a.w_)
                    v = a.x[((size_t)img * a.cin + ci) * HW + (size_t)yy * a.w_ + xx];
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(g, v, acc[t], 0, 0, 0);
            }
        }
    }
}

// VEC: rows of a multiple of four pixels, 16-byte aligned tensors.
template <bool VEC>
__global__ __launch_bounds__(kWgThreads) void conv3x3_wgrad_split_kernel(WgradSplitArgs a) {
    // the operands while the sums grow, the block's 64 x 64 x 9 sums afterwards
    union Shared {
        struct {
            uint4 xs[4][3][kWgOctets + 2][kWgStride];   // [row mod 4][term][octet, one more at either end]
            uint4 gs[2][3][kWgOctets][kWgStride];
        };
        float sums[kWgTile][kWgTile * 9];
    };
    __shared__ Shared lds;
    auto &xs = lds.xs;
    auto &gs = lds.gs;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int dy = wave >> 2, mh = (wave >> 1) & 1, nh = wave & 1;
    const int co0 = blockIdx.x * kWgTile, ci0 = blockIdx.y * kWgTile, slice = blockIdx.z;
    const int H = a.h, W = a.w_;
    const size_t HW = (size_t)H * W;
    const int c_begin = slice * a.cps, c_end = min(a.n_chunks, c_begin + a.cps);

    // Staging: the first 256 threads an octet of an input row each, the next
    // 256 one of dL/dz, 128 more one of the pixels beside the row.
    const int role = wave >> 2;                              // 0: input, 1: dL/dz, 2: edges (half of them)
    const int s_oct = tid & 3, s_ch = (tid >> 2) & 63;
    const int e_side = tid & 1, e_ch = (tid >> 1) & 63;
    const bool has_edge = tid >= 512 && tid < 640;
    float v[8];
    auto load_octet = [&](float (&v)[8], const float *row, int x0, bool ok) {
        if constexpr (VEC) {
            const bool lo = ok && x0 < W, hi = ok && x0 + 4 < W;
            const float4 p = *reinterpret_cast<const float4 *>(lo ? row + x0 : row);
            const float4 q = *reinterpret_cast<const float4 *>(hi ? row + x0 + 4 : row);
            v[0] = lo ? p.x : 0.0f; v[1] = lo ? p.y : 0.0f; v[2] = lo ? p.z : 0.0f; v[3] = lo ? p.w : 0.0f;
            v[4] = hi ? q.x : 0.0f; v[5] = hi ? q.y : 0.0f; v[6] = hi ? q.z : 0.0f; v[7] = hi ? q.w : 0.0f;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const bool in = ok && x0 + j < W;
                const float p = row[in ? x0 + j : 0];
                v[j] = in ? p : 0.0f;
            }
        }
    };
    // input row yy of a strip (zero outside the image)
    auto load_input = [&](float (&v)[8], int img, int strip, int yy) {
        const float *xi = a.x + (size_t)img * a.cin * HW;
        const int x0 = strip * kWgPixels;
        if (role == 0) {
            const bool ok = ci0 + s_ch < a.cin && yy >= 0 && yy < H;
            load_octet(v, xi + (ok ? (size_t)(ci0 + s_ch) * HW + (size_t)yy * W : 0), x0 + s_oct * 8, ok);
        } else if (has_edge) {
            const int xx = e_side ? x0 + kWgPixels : x0 - 1;
            const bool ok = ci0 + e_ch < a.cin && yy >= 0 && yy < H && xx >= 0 && xx < W;
            const float p = xi[ok ? (size_t)(ci0 + e_ch) * HW + (size_t)yy * W + xx : 0];
            v[0] = ok ? p : 0.0f;
        }
    };
    auto load_grad = [&](int img, int strip, int y) {
        if (role != 1) return;
        const bool ok = co0 + s_ch < a.cout;
        const float *gi = a.gz + (size_t)img * a.cout * HW;
        load_octet(v, gi + (ok ? (size_t)(co0 + s_ch) * HW + (size_t)y * W : 0), strip * kWgPixels + s_oct * 8, ok);
    };
    auto split_octet = [&](const float (&v)[8], uint4 (&t)[3]) {
        unsigned *h = &t[0].x, *m = &t[1].x, *l = &t[2].x;
        bool tiny = false;
#pragma unroll
        for (int j = 0; j < 8; j += 2) tiny |= split_pair(v[j], v[j + 1], h[j / 2], m[j / 2], l[j / 2]);
        // the first two pixels: every tap's octet holds one of them
        t[0].x = tiny ? kMarkPair : t[0].x;
    };
    auto store_input = [&](const float (&v)[8], int yy) {
        const int slot = (yy + 1) & 3;
        if (role == 0) {
            uint4 t[3];
            split_octet(v, t);
#pragma unroll
            for (int k = 0; k < 3; ++k) xs[slot][k][1 + s_oct][s_ch] = t[k];
        } else if (has_edge) {
            // the last pixel of the octet before, the first of the one after
            unsigned t[3];
            if (split_pair(e_side ? v[0] : 0.0f, e_side ? 0.0f : v[0], t[0], t[1], t[2])) t[0] = kMarkPair;
#pragma unroll
            for (int k = 0; k < 3; ++k)
                reinterpret_cast<unsigned *>(&xs[slot][k][e_side ? 1 + kWgOctets : 0][e_ch])[e_side ? 0 : 3] = t[k];
        }
    };
    auto store_grad = [&](int buf, bool negative) {
        if (role != 1) return;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = negative ? -v[j] : v[j];
        uint4 t[3];
        split_octet(v, t);
#pragma unroll
        for (int k = 0; k < 3; ++k) gs[buf][k][s_oct][s_ch] = t[k];
    };

    // counts negatively: every second pair of chunks
    const auto negative = [&](int c) { return ((c - c_begin) & 2) != 0; };
    int y = c_begin % H, strip = c_begin / H % a.strips, img = c_begin / H / a.strips;
    {
        // the first chunk, its loads all in flight
        float rows[3][8];
        load_grad(img, strip, y);
#pragma unroll
        for (int k = 0; k < 3; ++k) load_input(rows[k], img, strip, y - 1 + k);
        store_grad(0, false);
#pragma unroll
        for (int k = 0; k < 3; ++k) store_input(rows[k], y - 1 + k);
    }
    bool fresh = false;      // a chunk starts a strip: its input rows are not in the ring
    v16f acc[3], low[3];
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = low[t][r] = 0.0f;
    for (int c = c_begin; c < c_end; ++c) {
        const int buf = (c - c_begin) & 1;
        if (fresh) {
            for (int k = 0; k < 3; ++k) {
                load_input(v, img, strip, y - 1 + k);
                store_input(v, y - 1 + k);
            }
        }
        __syncthreads();
        // the next chunk: its dL/dz, and its last input row unless it starts a strip
        int y1 = y + 1, strip1 = strip, img1 = img;
        if (y1 == H) {
            y1 = 0;
            if (++strip1 == a.strips) {
                strip1 = 0;
                ++img1;
            }
        }
        const bool more = c + 1 < c_end;
        fresh = y1 == 0;
        if (more) {
            load_grad(img1, strip1, y1);
            if (!fresh) load_input(v, img, strip, y + 2);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < kWgPixels / 16; ++ks) {
            const int q = 2 * ks + (lane >> 5);
            v8bf g[3], b[3][3];   // [term], [tap][term]
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                g[k] = __builtin_bit_cast(v8bf, gs[buf][k][q][mh * 32 + (lane & 31)]);
                const uint4 *col = &xs[(y + dy) & 3][k][q][nh * 32 + (lane & 31)];
                const uint4 u = col[kWgStride];
                b[0][k] = __builtin_bit_cast(v8bf, shifted_left(u, col[0].w));
                b[1][k] = __builtin_bit_cast(v8bf, u);
                b[2][k] = __builtin_bit_cast(v8bf, shifted_right(u, col[2 * kWgStride].x));
            }
            constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int p = 0; p < 6; ++p)
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    v16f &d = p < 5 ? low[t] : acc[t];
                    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g[TA[p]], b[t][TB[p]], d, 0, 0, 0);
                }
        }
        if (more) {
            store_grad(buf ^ 1, negative(c + 1));
            if (!fresh) store_input(v, y + 2);
            if (negative(c) != negative(c + 1)) {
#pragma unroll
                for (int t = 0; t < 3; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[t][r] = -acc[t][r];
                        low[t][r] = -low[t][r];
                    }
            }
            if (fresh) __syncthreads();   // every wave is done with the old strip's rows
        }
        y = y1;
        strip = strip1;
        img = img1;
    }
    const bool flip = c_end > c_begin && negative(c_end - 1);
    bool bad = false;
    unsigned least = ~0u;
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[t][r] += low[t][r];
            acc[t][r] = flip ? -acc[t][r] : acc[t][r];
            bad |= !(fabsf(acc[t][r]) <= FLT_MAX);
            least = min(least, rank_of(acc[t][r]));
        }
    const int ci = ci0 + nh * 32 + (lane & 31);
    if (__any(bad || least < kTiny)) redo_wgrad_fp32(a, c_begin, c_end, co0 + mh * 32 + (lane & 31), ci, dy, acc);
    // through LDS: a row of the output is 64 x 9 consecutive values, a lane's are 9 apart
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int co = mh * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
#pragma unroll
        for (int t = 0; t < 3; ++t) lds.sums[co][(nh * 32 + (lane & 31)) * 9 + dy * 3 + t] = acc[t][r];
    }
    __syncthreads();
    float *o = a.out + (size_t)slice * a.cout * a.cin * 9 + ((size_t)co0 * a.cin + ci0) * 9;
    const int rows = min(kWgTile, a.cout - co0), run = min(kWgTile, a.cin - ci0) * 9;
#pragma unroll 1
    for (int r = wave; r < rows; r += kWgThreads / 64)
        for (int e = lane; e < run; e += 64) o[(size_t)r * a.cin * 9 + e] = lds.sums[r][e];
}

// How a convolution runs: the block tile, the tiling of the image, the K split.
struct SplitPlan {
    int wm, wn, tw, th, tiles_x, tiles_y, co_tiles, slices, cps;
    size_t part_floats;
    double us;   // the estimate below
};

// Estimated time (us), fitted to a sweep of (block tile, slices) over the layer
// shapes of the VGG-19 and StyleGAN2 networks on MI355X: a block's chunk takes
// a compute unit 5.1 us whether one or two blocks share it; the last round of
// blocks is partly hidden; ~6 us of launch, first loads and last stores; a
// split adds the sum kernel and its pass over the partial sums.  Its pick was
// within 6 % of the sweep's best on every shape (e.g. 512 -> 512 at 64 x 64:
// 2 x 2 waves in 4 slices, 98 us; unsplit 180 us).
double split_estimate_us(const SplitPlan &p, int n, size_t out_bytes) {
    const double blocks = (double)p.tiles_x * p.tiles_y * p.co_tiles * n * p.slices;
    const double rounds = blocks / kComputeUnits, full = std::ceil(rounds);
    double t = 6.0 + (rounds + 2.0 * full) / 3.0 * (p.cps * (p.wm == 1 ? 5.25 : 5.1) + 0.6);
    if (p.slices > 1) t += (double)(p.slices + 1) * out_bytes / 8.0e6 + 2.0;
    return t;
}

SplitPlan plan_split(int n, int cin, int h, int w, int cout) {
    SplitPlan best{};
    const int n_chunks = chunks_of(cin);
    const size_t out_bytes = (size_t)n * cout * h * w * sizeof(float);
    const int max_slices = std::max(1, std::min({kMaxSlices, n_chunks, 65535 / n}));
    for (int wm = 2; wm >= 1; --wm) {
        SplitPlan p{};
        p.wm = wm;
        p.wn = 4 / wm;
        p.tw = pick_tile_width(w);
        // 256-pixel tiles of 4 columns would need a 396-pixel halo tile
        if (p.wn == 4 && p.tw < 8) continue;
        p.th = 64 * p.wn / p.tw;
        p.tiles_x = (w + p.tw - 1) / p.tw;
        p.tiles_y = (h + p.th - 1) / p.th;
        p.co_tiles = (cout + 64 * wm - 1) / (64 * wm);
        for (int s = 1; s <= max_slices; ++s) {
            p.cps = (n_chunks + s - 1) / s;
            p.slices = (n_chunks + p.cps - 1) / p.cps;
            if (p.slices != s) continue;
            p.us = split_estimate_us(p, n, out_bytes);
            if (best.wm == 0 || p.us < 0.98 * best.us) best = p;
        }
    }
    best.part_floats = best.slices > 1 ? (size_t)best.slices * n * cout * h * w : 0;
    return best;
}

template <int WM, int WN>
void launch_split(const SplitArgs &s, const SplitPlan &p, hipStream_t st) {
    const dim3 grid((unsigned)(p.tiles_x * p.tiles_y), (unsigned)p.co_tiles, (unsigned)(s.c.n * p.slices));
    if (s.c.gate) hipLaunchKernelGGL((conv3x3_split_kernel<WM, WN, true>), grid, dim3(kThreads), 0, st, s);
    else hipLaunchKernelGGL((conv3x3_split_kernel<WM, WN, false>), grid, dim3(kThreads), 0, st, s);
}

int run_split(const char *what, ConvArgs a, const void *split, void *workspace, size_t workspace_bytes,
              hipStream_t st) {
    if (!conv_shape_ok(a.n, a.cin, a.h, a.w_, a.cout))
        return fail(SVBRDF_ESHAPE, "%s: n=%d cin=%d cout=%d height=%d width=%d", what, a.n, a.cin, a.cout, a.h, a.w_);
    if (a.cin < kKC)
        return fail(SVBRDF_ESHAPE, "%s: %d input channels, the split path takes %d or more", what, a.cin, kKC);
    if (a.act < SVBRDF_ACT_NONE || a.act > SVBRDF_ACT_LRELU)
        return fail(SVBRDF_EINVAL, "%s: unknown activation %d", what, a.act);
    if ((uintptr_t)split & 15u) return fail(SVBRDF_EINVAL, "%s: split weights must be 16-byte aligned", what);
    const SplitPlan p = plan_split(a.n, a.cin, a.h, a.w_, a.cout);
    const size_t need = p.part_floats * sizeof(float);
    if (need && (!workspace || workspace_bytes < need))
        return fail(SVBRDF_ESPACE, "%s: workspace of %zu bytes, this shape needs %zu "
                    "(svbrdf_conv3x3_split_workspace_bytes)", what, workspace ? workspace_bytes : (size_t)0, need);
    a.part = p.slices > 1 ? (float *)workspace : nullptr;
    a.tw = p.tw; a.th = p.th; a.tiles_x = p.tiles_x; a.slices = p.slices; a.cps = p.cps;
    const SplitArgs s{a, (const uint4 *)split};
    if (p.wm == 1) launch_split<1, 4>(s, p, st);
    else launch_split<2, 2>(s, p, st);
    if (p.slices > 1) launch_split_sum(a, st);
    return check_launch(what);
}

size_t split_floats(int k, int m) { return (size_t)chunks_of(k) * 9 * 3 * groups_of(m) * 64 * 4; }

}  // namespace

namespace svbrdf_internal {

WgradSplitPlan plan_wgrad_split(int n, int cin, int h, int w, int cout) {
    WgradSplitPlan p{};
    p.strips = (w + kWgPixels - 1) / kWgPixels;
    p.n_chunks = n * p.strips * h;
    p.co_tiles = (cout + kWgTile - 1) / kWgTile;
    p.ci_tiles = (cin + kWgTile - 1) / kWgTile;
    const double blocks = (double)p.co_tiles * p.ci_tiles, out_bytes = 36.0 * cin * cout;
    const int max_slices = std::max(1, std::min(256, p.n_chunks / 2));
    for (int s = 1; s <= max_slices; ++s) {
        const int cps = (p.n_chunks + s - 1) / s;
        if ((p.n_chunks + cps - 1) / cps != s) continue;   // no empty slice
        // measured: one block a compute unit at a time, a chunk 3.1 us, ~11 for
        // the launch, the first loads and the last stores, then the slices' sum
        double t = std::ceil(blocks * s / kComputeUnits) * (cps * 3.1 + 3.0) + 8.0;
        if (s > 1) t += (s + 1) * out_bytes / 5.3e6 + 1.5;
        if (s == 1 || t < 0.98 * p.us) {
            p.us = t;
            p.slices = s;
            p.cps = cps;
        }
    }
    return p;
}

void launch_wgrad_split(const WgradSplitPlan &p, const float *x, const float *grad_z, int n, int cin, int h, int w,
                        int cout, float *out, hipStream_t s) {
    const WgradSplitArgs a{x, grad_z, out, n, cin, cout, h, w, p.strips, p.n_chunks, p.cps};
    const dim3 grid((unsigned)p.co_tiles, (unsigned)p.ci_tiles, (unsigned)p.slices);
    const bool vec = w % 4 == 0 && (((uintptr_t)x | (uintptr_t)grad_z) & 15u) == 0;
    if (vec) hipLaunchKernelGGL(conv3x3_wgrad_split_kernel<true>, grid, dim3(kWgThreads), 0, s, a);
    else hipLaunchKernelGGL(conv3x3_wgrad_split_kernel<false>, grid, dim3(kWgThreads), 0, s, a);
}

}  // namespace svbrdf_internal

extern "C" {

// Where this path is taken.  Below ~2 GFLOP a call is bound by its launches
// and first loads, not the matrix cores, and the fp32 kernel's finer chunks
// win (graph-timed, fp32 / split without the weights' 6-8 us: 64 -> 64 at 64^2
// 12.5 / 14.1 us, 128 -> 128 at 32^2 13.1 / 15.1, 512 -> 512 at 16^2 25.5 /
// 22.6; above it 512 -> 512 at 32^2 64.7 / 34.9, 512 -> 512 at 64^2 189 / 98,
// 9 x 64 -> 64 at 256^2 387 / 224).  With fewer than 32 input channels the
// 16-channel chunks are mostly padding, and the short sums are no more exact
// than fp32's.
int svbrdf_conv3x3_split_preferred(int n, int cin, int height, int width, int cout) {
    if (!conv_shape_ok(n, cin, height, width, cout)) return 0;
    return cout > kDirectMaxCout && cin >= 32 && 18.0 * n * cin * cout * height * width >= 2.0e9;
}

// Where each call also splits the packed weights it is given: 90 bytes for
// each pair of channels, 12 us a million pairs and 18 above three million (past
// the caches), at least 3.7, and 3 for the launch. Layers of many channels on few pixels are mostly that pass
// (fp32 / split with it, us: 4096 -> 4096 at 4^2 197 / 487, 2048 -> 2048 at 8^2
// 61 / 124, 9 x 512 -> 512 at 8^2 42 / 45; 512 -> 512 at 22^2 46 / 38). Over 275
// shapes of 32 to 4096 channels between 2 and 12 GFLOP this line takes one that
// is slower by more than 2 % (256 -> 512 at 32^2, 35 / 37) and leaves 14 that
// would be faster by more than 3 %, none of at most 512 channels.
int svbrdf_conv3x3_split_packed_preferred(int n, int cin, int height, int width, int cout) {
    if (!svbrdf_conv3x3_split_preferred(n, cin, height, width, cout)) return 0;
    const double weights = (double)cin * cout;
    const double pass = 3.0 + std::max(3.7, weights * (weights < 3.0e6 ? 1.2e-5 : 1.8e-5));
    constexpr double kLaunch = 4.0;   // in split_estimate_us, not in conv_us
    return plan_split(n, cin, height, width, cout).us + pass < conv_us(n, cin, height, width, cout) + kLaunch;
}

size_t svbrdf_conv3x3_split_weights_bytes(int cin, int cout) {
    if (cin < 1 || cout < 1 || cin > kMaxChannels || cout > kMaxChannels) return 0;
    // the split weights, then room for a demodulation factor per channel of either side
    return (split_floats(cin, cout) + std::max(cin, cout)) * sizeof(float);
}

int svbrdf_conv3x3_pack_split(const float *weight, int cout, int cin, const float *style, float scale, int demodulate,
                              int transpose, void *split, void *stream) {
    const char *what = "svbrdf_conv3x3_pack_split";
    if (!weight || !split) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    if (cout < 1 || cin < 1 || cout > kMaxChannels || cin > kMaxChannels)
        return fail(SVBRDF_ESHAPE, "%s: cout=%d cin=%d outside [1, %d]", what, cout, cin, kMaxChannels);
    if ((uintptr_t)split & 15u) return fail(SVBRDF_EINVAL, "%s: split weights must be 16-byte aligned", what);
    hipStream_t s = (hipStream_t)stream;
    const int m = transpose ? cin : cout, k = transpose ? cout : cin;
    if (k < kKC) return fail(SVBRDF_ESHAPE, "%s: %d input channels, the split path takes %d or more", what, k, kKC);
    float *factor = nullptr;
    if (demodulate) {
        factor = (float *)split + split_floats(k, m);
        hipLaunchKernelGGL(split_factor_kernel, dim3((unsigned)cout), dim3(kThreads), 0, s, weight, cin, style, scale,
                           factor);
        if (int rc = check_launch(what)) return rc;
    }
    const dim3 grid((unsigned)groups_of(m), (unsigned)chunks_of(k));
    if (transpose)
        hipLaunchKernelGGL(split_pack_kernel<kTransposed>, grid, dim3(kThreads), 0, s, weight, m, k, style, scale,
                           (const float *)factor, (uint4 *)split);
    else
        hipLaunchKernelGGL(split_pack_kernel<kNatural>, grid, dim3(kThreads), 0, s, weight, m, k, style, scale,
                           (const float *)factor, (uint4 *)split);
    return check_launch(what);
}

int svbrdf_conv3x3_split_packed(const float *packed, int cin, int cout, void *split, void *stream) {
    const char *what = "svbrdf_conv3x3_split_packed";
    if (!packed || !split) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    if (cout < 1 || cin < 1 || cout > kMaxChannels || cin > kMaxChannels)
        return fail(SVBRDF_ESHAPE, "%s: cout=%d cin=%d outside [1, %d]", what, cout, cin, kMaxChannels);
    if ((uintptr_t)split & 15u) return fail(SVBRDF_EINVAL, "%s: split weights must be 16-byte aligned", what);
    if (cin < kKC) return fail(SVBRDF_ESHAPE, "%s: %d input channels, the split path takes %d or more", what, cin, kKC);
    const dim3 grid((unsigned)groups_of(cout), (unsigned)chunks_of(cin));
    hipLaunchKernelGGL(split_pack_kernel<kPacked>, grid, dim3(kThreads), 0, (hipStream_t)stream, packed, cout, cin,
                       (const float *)nullptr, 1.0f, (const float *)nullptr, (uint4 *)split);
    return check_launch(what);
}

size_t svbrdf_conv3x3_split_workspace_bytes(int n, int cin, int height, int width, int cout) {
    if (!conv_shape_ok(n, cin, height, width, cout) || cin < kKC) return 0;
    return plan_split(n, cin, height, width, cout).part_floats * sizeof(float);
}

int svbrdf_conv3x3_split(const float *x, int n, int cin, int height, int width, const void *split, int cout,
                         const float *bias, const float *noise, float noise_strength, int activation, float *y,
                         void *workspace, size_t workspace_bytes, void *stream) {
    const char *what = "svbrdf_conv3x3_split";
    if (!x || !split || !y) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    ConvArgs a{};
    a.x = x; a.bias = bias; a.noise = noise; a.noise_strength = noise_strength; a.act = activation;
    a.y = y; a.n = n; a.cin = cin; a.cout = cout; a.h = height; a.w_ = width;
    return run_split(what, a, split, workspace, workspace_bytes, (hipStream_t)stream);
}

// Where a tile holds whole 2 x 2 windows and all of K: 32 columns (images wider
// than 16), unsplit. The layer before VGG's first pooling (9 x 64 x 256^2) then
// writes its scaled copy and 38 MB of averages instead of 151 MB that a pooling
// kernel reads again: 309 + 44 us -> 296; the second one 211 + 15 -> 214.
int svbrdf_conv3x3_split_pools(int n, int cin, int height, int width, int cout) {
    if (!svbrdf_conv3x3_split_preferred(n, cin, height, width, cout) || height < 2) return 0;
    const SplitPlan p = plan_split(n, cin, height, width, cout);
    return p.slices == 1 && p.tw == 32;
}

int svbrdf_conv3x3_pooled(const float *x, int n, int cin, int height, int width, const void *split, int cout,
                          const float *bias, const float *noise, float noise_strength, int activation, float *y,
                          float *tap, float tap_scale, float *pool, void *stream) {
    const char *what = "svbrdf_conv3x3_pooled";
    if (!x || !split || !pool) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    if (!svbrdf_conv3x3_split_pools(n, cin, height, width, cout))
        return fail(SVBRDF_ESHAPE, "%s: n=%d cin=%d cout=%d height=%d width=%d (svbrdf_conv3x3_split_pools)", what, n,
                    cin, cout, height, width);
    ConvArgs a{};
    a.x = x; a.bias = bias; a.noise = noise; a.noise_strength = noise_strength; a.act = activation;
    a.y = y; a.tap = tap; a.tap_scale = tap_scale; a.pool = pool;
    a.n = n; a.cin = cin; a.cout = cout; a.h = height; a.w_ = width;
    return run_split(what, a, split, nullptr, 0, (hipStream_t)stream);
}

int svbrdf_conv3x3_tapped(const float *x, int n, int cin, int height, int width, const float *packed,
                          const void *split, int cout, const float *bias, const float *noise, float noise_strength,
                          int activation, float *y, float *tap, float tap_scale, void *workspace,
                          size_t workspace_bytes, void *stream) {
    const char *what = "svbrdf_conv3x3_tapped";
    if (!x || (!packed && !split) || !y || !tap) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    ConvArgs a{};
    a.x = x; a.w = packed; a.bias = bias; a.noise = noise; a.noise_strength = noise_strength; a.act = activation;
    a.y = y; a.tap = tap; a.tap_scale = tap_scale; a.n = n; a.cin = cin; a.cout = cout; a.h = height; a.w_ = width;
    return split ? run_split(what, a, split, workspace, workspace_bytes, (hipStream_t)stream)
                 : run_conv(what, a, workspace, workspace_bytes, (hipStream_t)stream);
}

int svbrdf_conv3x3_input_grad_split(const float *grad_y, const float *y, int activation, int n, int cout, int height,
                                    int width, const void *split_t, int cin, float *grad_x, void *workspace,
                                    size_t workspace_bytes, void *stream) {
    const char *what = "svbrdf_conv3x3_input_grad_split";
    if (!grad_y || !y || !split_t || !grad_x) return fail(SVBRDF_EINVAL, "%s: null pointer argument", what);
    if (activation < SVBRDF_ACT_NONE || activation > SVBRDF_ACT_LRELU)
        return fail(SVBRDF_EINVAL, "%s: unknown activation %d", what, activation);
    const ConvArgs a = input_grad_args(grad_y, y, activation, n, cout, height, width, cin, grad_x);
    return run_split(what, a, split_t, workspace, workspace_bytes, (hipStream_t)stream);
}

}  // extern "C"
