// mbrec_unet.hip -- learned warm start: a 4-level convolutional U-Net that maps
// the back-projected image A^T y to an initial NNLS estimate.
//
// No counterpart in the reference (its NNLS loops always start from zero,
// nnls_L2_less.m:28-29); the estimate enters the solver through the initial
// image of the warm-start form of rec_nn_with_L2_reg (rec_nn_with_L2_reg.m:41).
//
// Architecture (base width c, all 3x3 convolutions with zero padding, ReLU):
//   enc1 1->c, c->c | pool | enc2 c->2c, 2c->2c | pool | enc3 2c->4c, 4c->4c | pool
//   bottleneck 4c->8c, 8c->8c | up+cat enc3 | 12c->4c, 4c->4c | up+cat enc2 | 6c->2c, 2c->2c
//   | up+cat enc1 | 3c->c, c->c | 1x1 head c->1 (linear)
// Pooling is a 2x2 average, upsampling nearest-neighbour.  Each image is scaled
// by s = rms(A^T y) before the network and the output is multiplied by s.
//
// Numerics: activations and activation gradients are stored in bfloat16
// (round to nearest even) in pixel-major / channel-minor order; every 3x3
// convolution with >= 32 input channels runs on the matrix cores
// (v_mfma_f32_32x32x16_bf16, FP32 accumulation) as an implicit GEMM over
// (pixels x output channels x 9*input channels); its input gradient is the same
// kernel with the flipped, transposed filter, and its filter gradient an
// implicit GEMM over pixels.  The first convolution (one input channel), the
// 1x1 head, pooling, upsampling, the loss and Adam run on the vector ALUs in
// FP32.  Master weights and Adam moments are FP32.
#include "mbrec_internal.h"

#include <cmath>
#include <algorithm>
#include <type_traits>

namespace mbrec {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ __forceinline__ float bf2f(uint16_t h)
{
    union { uint32_t u; float f; } c;
    c.u = (uint32_t)h << 16;
    return c.f;
}

__host__ __device__ __forceinline__ uint16_t f2bf(float f)
{
    union { uint32_t u; float f; } c;
    c.f = f;
    uint32_t u = c.u;
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// ---------------------------------------------------------------------------
// 3x3 convolution, implicit GEMM on the matrix cores.
// y[p][yo + co] = act(bias[co] + sum_{t, ci} x[p + shift(t)][ci] * w[co][t][ci])
//
// The batch is one wide image: virtual column X = n Wp + w with Wp - W >= 1 columns of
// zeros between images (their outputs are not stored), so that the 32-pixel fragments of a
// narrow level run across images instead of ending in padding (W = 50: 4 % instead of 28 %),
// and Wp - W is even for an even W, which keeps 2 x 2 pixel blocks inside a fragment.
//
// Workgroup = 32 columns x 8 rows x 32 NB output channels (NB: conv_launch); wave = 2 rows.  Per 32 input
// channels the 10 x 34 input pixels and the 9 taps' filters go memory -> LDS (16-byte loads
// with the LDS destination; pixels outside read a zero block).  Products are 32x32x16 with
// A = filters (rows = output channels) and B = pixels (columns): a pixel fragment of input row
// h serves the output rows h - 1, h, h + 1, so 6 NB products take 4 + 3 NB fragment reads, and
// the accumulators of a lane are 4 consecutive channels of one pixel (8-byte stores).  The
// 16-byte slots of a pixel are permuted by its column ((col >> 1) & 3) so that the 8 lanes
// of an LDS read cycle touch all banks; rows only change an immediate offset.
// 43 KB of LDS and 124 registers (NB = 1): three workgroups per CU, one staging while the others multiply.  Tiles
// of 16 rows x 64 channels (78 KB, 254 registers, four spilled) read less LDS per product but left CUs idle on small
// images and waited more on large ones: the network on one image of 152^2 0.436 -> 0.192 ms (0.392 with the
// direct form below), 8 x 400^2 0.96 -> 0.76, 64 x 400^2 5.66 -> 5.22 ms.  A sum's K order is the same for both.
// The channels of a concatenation come straight from its two sources (the first at half
// resolution where `up`: nearest-neighbour upsampling without a copy).
// Measured: the network on 64 images of 400^2 (3.3 TFLOP) 27.1 -> 5.2 ms (122 -> 635 TFLOP/s)
// against a direct form whose waves read both operands from global memory for every product, with
// separate pooling, upsampling and head passes.  The levels of 32 channels are bound by HBM
// (0.65 GB per tensor at 64 x 400^2), the others by LDS reads and staging waits.
//
// EPI (epilogue):
//   kRelu   y = relu(acc + bias); with yp also its 2 x 2 average pool
//   kHead   as kRelu (y may be null), and the 1x1 head: on / out
//   kGrad   y = acc where the mask m > 0 (m may be null)
//   kGradUp channels < n_low: sum over the 2 x 2 block (upsampling backward) where the mask
//           mp > 0, to yp at half resolution; the others to y (channel - n_low)
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

enum { kRelu, kHead, kGrad, kGradUp };
constexpr int kCvCols = 32, kCvRows = 8;      // output tile of a workgroup
constexpr int staged_slots(int rows) { return (rows + 2) * (kCvCols + 2) * 4; }   // 16-byte slots of 32 channels, with the halo

__device__ __attribute__((aligned(16))) const uint16_t g_zero_slot[8] = {0, 0, 0, 0, 0, 0, 0, 0};

struct ConvSrc {
    const uint16_t *p;
    int cs, co, up;       // channels per pixel, first channel, 1: half resolution
};

struct ConvArgs {
    ConvSrc src[2];       // channels [0, split) and [split, Cin)
    int split, Cin, Cout;
    const uint16_t *w;
    const float *bias;
    uint16_t *y;
    int ys, yo;
    const uint16_t *m;
    int ms, mo;
    uint16_t *yp;
    const uint16_t *mp;
    int n_low;
    const float *hw, *hb, *s;
    float *on, *out;
    int N, H, W, Wp, tiles_x, ntiles, ncot, tile0;
};

// memory -> LDS, 16 bytes per lane; dst is the wave's base
__device__ __forceinline__ void copy_to_lds(const uint16_t *src, uint16_t *dst)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                     (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}

// 16-byte slot `slot` (8 channels) of virtual column X, row h: its index from c.p + c.co, or -1 outside the
// images (T: int below 2^31 slots, 32 GB of input, else 64 bits)
template <typename T = int>
__device__ __forceinline__ T conv_slot(const ConvSrc &c, int X, int h, int slot, int N, int H, int W, int Wp)
{
    if (X < 0 || h < 0 || h >= H) return -1;
    const int n = X / Wp, w = X - n * Wp;
    if (n >= N || w >= W) return -1;
    const int px = c.up ? (n * (H / 2) + h / 2) * (W / 2) + w / 2 : (n * H + h) * W + w;
    return (T)px * (c.cs / 8) + slot;
}

template <int NB, int EPI, typename T>
__global__ __launch_bounds__(256, NB == 1 ? 3 : 2) void k_conv3(const ConvArgs a)
{
    constexpr int CO = 32 * NB, R = kCvRows / 4;                                // R: rows of a wave
    constexpr int IN = staged_slots(kCvRows), INIT = (IN + 255) / 256;   // 16-byte slots of the staged input, per thread
    __shared__ __attribute__((aligned(16))) uint16_t s_in[INIT * 256 * 8];
    __shared__ __attribute__((aligned(16))) uint16_t s_w[9 * CO * 32];
    // blocks of one XCD (every eighth) take the channel tiles of a pixel tile in a row
    const int k = blockIdx.x >> 3, ct = k % a.ncot, sp = a.tile0 + (k / a.ncot) * 8 + (blockIdx.x & 7);
    if (sp >= a.ntiles) return;   // whole workgroup, before any barrier
    const int ty = sp / a.tiles_x, tx = sp - ty * a.tiles_x;
    const int X0 = tx * kCvCols, h0 = ty * kCvRows, co0 = ct * CO;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, hl = lane >> 5;
    const int H = a.H, W = a.W, Cin = a.Cin;

    // filter source of this thread: output channel and slot fixed, tap = it (NB = 2) or 2 it + tid / 128 (NB = 1)
    const int wco = (tid >> 2) % CO, wt0 = (tid >> 2) / CO;
    const uint16_t *wsrc = a.w + ((size_t)(co0 + wco) * 9 + wt0) * Cin + 8 * ((tid & 3) ^ ((wco >> 1) & 3));

    f32x16 acc[R][NB];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[r][nb][i] = 0.0f;

    int pa[3];   // byte offset of this lane's pixel fragment (slot half 0) per column shift
#pragma unroll
    for (int dx = 0; dx < 3; ++dx)
        pa[dx] = (R * wv * (kCvCols + 2) + j + dx) * 64 + ((hl ^ (((j + dx) >> 1) & 3)) << 4);
    const int wa = j * 64 + ((hl ^ ((j >> 1) & 3)) << 4);
    const bool live = h0 + R * wv < H;

    for (int sidx = 0; sidx < 2; ++sidx) {
        const int nch = sidx ? Cin - a.split : a.split;
        if (nch <= 0) continue;
        T slot[INIT];
#pragma unroll
        for (int it = 0; it < INIT; ++it) {
            const int e = it * 256 + tid, px = e >> 2, row = px / (kCvCols + 2), col = px - row * (kCvCols + 2);
            slot[it] = e < IN ? conv_slot<T>(a.src[sidx], X0 + col - 1, h0 + row - 1, (e & 3) ^ ((col >> 1) & 3), a.N, H, W,
                                             a.Wp)
                                 : -1;
        }
        const uint16_t *base = a.src[sidx].p + a.src[sidx].co;
        for (int c0 = 0; c0 < nch; c0 += 32) {
            __syncthreads();   // the previous chunk is no longer read
#pragma unroll
            for (int it = 0; it < INIT; ++it)
                copy_to_lds(slot[it] >= 0 ? base + c0 + (size_t)(std::make_unsigned_t<T>)slot[it] * 8 : g_zero_slot,
                            s_in + (it * 256 + wv * 64) * 8);
#pragma unroll
            for (int it = 0; it < (9 * CO * 4 + 255) / 256; ++it)
                if (it * 256 + wv * 64 < 9 * CO * 4)
                    copy_to_lds(wsrc + (size_t)it * (64 / CO) * Cin, s_w + (it * 256 + wv * 64) * 8);
            wsrc += 32;
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
            __syncthreads();
            if (live) {
                const char *bi = reinterpret_cast<const char *>(s_in), *bw = reinterpret_cast<const char *>(s_w);
#pragma unroll
                for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) {
                        bf16x8 fw[3][NB];
#pragma unroll
                        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                            for (int nb = 0; nb < NB; ++nb)
                                fw[dy][nb] = *reinterpret_cast<const bf16x8 *>(bw + (wa ^ (kh << 5)) +
                                                                               ((3 * dy + dx) * CO + 32 * nb) * 64);
#pragma unroll
                        for (int row = 0; row < R + 2; ++row) {
                            const bf16x8 fx = *reinterpret_cast<const bf16x8 *>(bi + (pa[dx] ^ (kh << 5)) +
                                                                                row * (kCvCols + 2) * 64);
#pragma unroll
                            for (int dy = 0; dy < 3; ++dy) {
                                const int r = row - dy;
                                if (r < 0 || r >= R) continue;
#pragma unroll
                                for (int nb = 0; nb < NB; ++nb)
                                    acc[r][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[dy][nb], fx, acc[r][nb], 0,
                                                                                         0, 0);
                            }
                        }
                    }
            }
        }
    }
    if (!live) return;   // no barriers below

    // lane: column X, output channels 32 nb + 8 q + 4 hl + i of acc[r][nb][4 q + i]
    const int X = X0 + j, n = X / a.Wp, w = X - n * a.Wp;
    const bool pv = n < a.N && w < W;
    const bool low = EPI == kGradUp && co0 < a.n_low;
#pragma unroll
    for (int rp = 0; rp < R; rp += 2) {
        float head[2] = {0.0f, 0.0f};
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int co = co0 + 32 * nb + 8 * q + 4 * hl;
                u16x4 o[2];
#pragma unroll
                for (int dr = 0; dr < 2; ++dr) {
                    const int h = h0 + R * wv + rp + dr;
                    const bool ok = pv && h < H;
                    const size_t p = ((size_t)n * H + h) * W + w;
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v[i] = acc[rp + dr][nb][4 * q + i];
                        if constexpr (EPI == kRelu || EPI == kHead) v[i] = fmaxf(v[i] + (a.bias ? a.bias[co + i] : 0.0f), 0.0f);
                    }
                    if constexpr (EPI == kGrad) {
                        if (a.m && ok) {
                            const u16x4 mv = *reinterpret_cast<const u16x4 *>(a.m + p * a.ms + a.mo + co);
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (!(bf2f(mv[i]) > 0.0f)) v[i] = 0.0f;
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[dr][i] = f2bf(v[i]);
                    if constexpr (EPI == kHead) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) head[dr] = fmaf(a.hw[co + i], bf2f(o[dr][i]), head[dr]);
                    }
                    if (ok && !low && (EPI != kHead || a.y))
                        *reinterpret_cast<u16x4 *>(a.y + p * a.ys + a.yo + co - (EPI == kGradUp ? a.n_low : 0)) = o[dr];
                }
                if constexpr (EPI == kRelu || EPI == kGradUp) {
                    if (EPI == kRelu ? a.yp != nullptr : low) {   // uniform
                        const int h = h0 + R * wv + rp;
                        const bool ok = pv && h < H && !(j & 1);
                        const int nl = EPI == kRelu ? a.Cout : a.n_low;
                        const size_t pl = (((size_t)n * (H / 2) + h / 2) * (W / 2) + w / 2) * nl + co;
                        u16x4 mv = {0, 0, 0, 0}, ov;
                        if (EPI == kGradUp && ok) mv = *reinterpret_cast<const u16x4 *>(a.mp + pl);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float v00 = bf2f(o[0][i]), v10 = bf2f(o[1][i]);
                            const float v01 = __shfl_xor(v00, 1), v11 = __shfl_xor(v10, 1);
                            const float t = ((v00 + v01) + v10) + v11;
                            if constexpr (EPI == kRelu) ov[i] = f2bf(0.25f * t);
                            else ov[i] = f2bf(bf2f(mv[i]) > 0.0f ? t : 0.0f);
                        }
                        if (ok) *reinterpret_cast<u16x4 *>(a.yp + pl) = ov;
                    }
                }
            }
        if constexpr (EPI == kHead) {
#pragma unroll
            for (int dr = 0; dr < 2; ++dr) {
                const float v = a.hb[0] + (head[dr] + __shfl_xor(head[dr], 32));
                const int h = h0 + R * wv + rp + dr;
                if (pv && h < H && hl == 0) {
                    const size_t p = ((size_t)n * H + h) * W + w;
                    if (a.on) a.on[p] = v;
                    if (a.out) a.out[p] = v * a.s[n];
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// filter and bias gradient of a 3x3 convolution (implicit GEMM over pixels):
// dw[co][t][ci] = sum_p g[p][co] * x[p + shift(t)][ci],  db[co] = sum_p g[p][co]
//
// Workgroup = 32 output x 32 input channels, all nine taps (144 accumulators per lane), and
// every nsplit-th tile of 32 columns x 16 rows; wave = 4 rows.  The tile of g and of x (with
// its halo) go memory -> LDS as in the convolution; pixels are the product's inner dimension,
// so the fragments are read transposed (ds_read_b64_tr_b16), which also makes the taps'
// column shifts plain addresses.  A row fragment of x serves three rows of g: 36 products per
// 22 fragments.  The bias is one more product with a fragment of ones (first channel tile).
// The waves' sums are joined in LDS and written as one partial per workgroup, summed in
// order by k_wgrad_sum: no atomics.  Measured at 400^2 x 8: 0.84 + 0.11 ms per training pass,
// against 10.8 ms for a kernel per tap with 2-byte loads and FP32 atomics and a separate bias pass
// (the whole pass 20.1 -> 3.7 ms).
// ---------------------------------------------------------------------------
constexpr int kWgRows = 16;                      // rows of a tile
constexpr int kWgIn = staged_slots(kWgRows), kWgInIt = (kWgIn + 255) / 256;
constexpr int kWgG = kWgRows * kCvCols * 4;      // 16-byte slots of the staged g tile
constexpr int kWgPart = 9 * 1024 + 32;           // floats of a partial: taps [9][16][64 lanes], bias [32]

struct WgradArgs {
    ConvSrc g, src[2];
    int split, Cin, Cout;
    float *part;
    int N, H, W, Wp, tiles_x, ntiles, npair, nsplit;
};

__device__ __forceinline__ bf16x8 read_tr(const uint16_t *p)
{
    typedef __attribute__((address_space(3))) s16x4 *lds_t;
    union { s16x4 h[2]; bf16x8 v; } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)const_cast<uint16_t *>(p));
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)const_cast<uint16_t *>(p + 4 * 32));   // four pixels on
    return u.v;
}

__global__ __launch_bounds__(256, 2) void k_conv3_wgrad(const WgradArgs a)
{
    // one array: the staged tiles, then the waves' accumulators
    __shared__ __attribute__((aligned(16))) uint16_t s_all[(kWgInIt * 256 + kWgG) * 8];
    uint16_t *s_in = s_all, *s_g = s_all + kWgInIt * 256 * 8;
    static_assert(sizeof(float) * 2 * 9 * 1024 <= sizeof(uint16_t) * (kWgInIt * 256 + kWgG) * 8, "two waves' accumulators");
    const int k = blockIdx.x >> 3, pair = k % a.npair, split = (k / a.npair) * 8 + (blockIdx.x & 7);
    if (split >= a.nsplit) return;   // whole workgroup, before any barrier
    const int nci = a.Cin / 32, co0 = (pair / nci) * 32, ci0 = (pair % nci) * 32;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool bias = ci0 == 0;
    ConvSrc xs = ci0 < a.split ? a.src[0] : a.src[1], gs = a.g;
    xs.co += ci0 < a.split ? ci0 : ci0 - a.split;
    gs.co += co0;
    // this lane's source of a transposed read: pixel (of 16), channel group
    const int tro = (8 * (lane >> 5) + ((lane & 15) >> 2)) * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;

    f32x16 acc[9], accb;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        accb[i] = 0.0f;
#pragma unroll
        for (int t = 0; t < 9; ++t) acc[t][i] = 0.0f;
    }
    bf16x8 one;
#pragma unroll
    for (int i = 0; i < 8; ++i) one[i] = (__bf16)1.0f;

    for (int sp = split; sp < a.ntiles; sp += a.nsplit) {
        const int ty = sp / a.tiles_x, tx = sp - ty * a.tiles_x;
        const int X0 = tx * kCvCols, h0 = ty * kWgRows;
        __syncthreads();   // the previous tile is no longer read
#pragma unroll
        for (int it = 0; it < kWgInIt; ++it) {
            const int e = it * 256 + tid, px = e >> 2, row = px / (kCvCols + 2), col = px - row * (kCvCols + 2);
            const int q = e < kWgIn ? conv_slot(xs, X0 + col - 1, h0 + row - 1, e & 3, a.N, a.H, a.W, a.Wp) : -1;
            copy_to_lds(q >= 0 ? xs.p + xs.co + (size_t)(unsigned)q * 8 : g_zero_slot, s_in + (it * 256 + wv * 64) * 8);
        }
#pragma unroll
        for (int it = 0; it < kWgG / 256; ++it) {
            const int e = it * 256 + tid, px = e >> 2;
            const int q = conv_slot(gs, X0 + (px & 31), h0 + (px >> 5), e & 3, a.N, a.H, a.W, a.Wp);
            copy_to_lds(q >= 0 ? gs.p + gs.co + (size_t)(unsigned)q * 8 : g_zero_slot, s_g + (it * 256 + wv * 64) * 8);
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
        __syncthreads();
        if (h0 + 4 * wv < a.H) {
#pragma unroll
            for (int ch = 0; ch < 2; ++ch) {
                bf16x8 fg[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    fg[r] = read_tr(s_g + ((4 * wv + r) * kCvCols + 16 * ch) * 32 + tro);
                if (bias) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg[r], one, accb, 0, 0, 0);
                }
#pragma unroll
                for (int row = 0; row < 6; ++row)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) {
                        const bf16x8 fx = read_tr(s_in + ((4 * wv + row) * (kCvCols + 2) + 16 * ch + dx) * 32 + tro);
#pragma unroll
                        for (int dy = 0; dy < 3; ++dy) {
                            const int r = row - dy;
                            if (r < 0 || r > 3) continue;
                            acc[3 * dy + dx] =
                                __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg[r], fx, acc[3 * dy + dx], 0, 0, 0);
                        }
                    }
            }
        }
    }
    // waves 2, 3 -> 0, 1, then 1 -> 0
    float *red = reinterpret_cast<float *>(s_all);
#pragma unroll
    for (int step = 2; step >= 1; step >>= 1) {
        __syncthreads();
        if (wv >= step && wv < 2 * step) {
            float *dst = red + (wv - step) * 9 * 1024 + lane;
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) dst[(t * 16 + i) * 64] = acc[t][i];
        }
        __syncthreads();
        if (wv < step) {
            const float *src = red + wv * 9 * 1024 + lane;
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[t][i] += src[(t * 16 + i) * 64];
        }
    }
    __syncthreads();
    if (bias && (lane & 31) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) red[wv * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)] = accb[i];
    }
    __syncthreads();
    float *dst = a.part + (size_t)(pair * a.nsplit + split) * kWgPart;
    if (bias && tid < 32) dst[9 * 1024 + tid] = (red[tid] + red[32 + tid]) + (red[64 + tid] + red[96 + tid]);
    if (wv == 0) {
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) dst[(t * 16 + i) * 64 + lane] = acc[t][i];
    }
}

// sums the nsplit partials of every channel pair: workgroup = 32 values x 8 runs of splits;
// blockIdx.x = 0 .. 287 taps, 288 the bias (of the pairs with ci0 = 0)
__global__ __launch_bounds__(256) void k_wgrad_sum(const float *__restrict__ part, float *__restrict__ dw,
                                                   float *__restrict__ db, int Cin, int nsplit)
{
    const int pair = blockIdx.y, nci = Cin / 32, co0 = (pair / nci) * 32, ci0 = (pair % nci) * 32;
    if (blockIdx.x == 288 && ci0) return;   // whole workgroup
    const int v = threadIdx.x & 31, run = threadIdx.x >> 5;
    const int e = blockIdx.x * 32 + v;
    const float *src = part + (size_t)pair * nsplit * kWgPart + e;
    float s = 0.0f;
#pragma unroll 8
    for (int k = run; k < nsplit; k += 8) s += src[(size_t)k * kWgPart];
    __shared__ float red[8][32];
    red[run][v] = s;
    __syncthreads();
    if (run) return;
#pragma unroll
    for (int k = 1; k < 8; ++k) s += red[k][v];
    if (e >= 9 * 1024) {
        db[co0 + v] = s;
        return;
    }
    const int t = e >> 10, i = (e >> 6) & 15, l = e & 63;
    dw[((size_t)(co0 + 8 * (i >> 2) + 4 * (l >> 5) + (i & 3)) * 9 + t) * Cin + ci0 + (l & 31)] = s;
}

// ---------------------------------------------------------------------------
// per-image scale s_b = sqrt(mean(in_b^2)) (tiny floor): sums of kScaleParts runs of an image
// (one workgroup per image left most CUs idle: 71 us at 400^2 whatever the batch), then s
// ---------------------------------------------------------------------------
constexpr int kScaleParts = 32;

__device__ __forceinline__ double block_sum_256(double v)
{
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) v += __shfl_xor(v, k);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void k_image_sumsq(const float *__restrict__ in, double *__restrict__ part, int HW)
{
    const float *src = in + (size_t)blockIdx.y * HW;
    double acc = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < HW; i += kScaleParts * 256) acc += (double)src[i] * src[i];
    acc = block_sum_256(acc);
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * kScaleParts + blockIdx.x] = acc;
}

__global__ void k_image_scale(const double *__restrict__ part, float *__restrict__ s, int B, int HW)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < kScaleParts; ++k) acc += part[(size_t)b * kScaleParts + k];
    s[b] = (float)fmax(sqrt(acc / HW), 1e-30);
}

// ---------------------------------------------------------------------------
// first convolution (1 input channel, C outputs), FP32, of the normalised input in / s:
// y[p][co] = relu(b + sum_t w[co][t] in_n[p+shift(t)]); in_n (may be null) keeps in / s
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_conv_first(const float *__restrict__ x, const float *__restrict__ s,
                                                    float *__restrict__ in_n, const float *__restrict__ w,
                                                    const float *__restrict__ b, uint16_t *__restrict__ y, int N,
                                                    int H, int W, int C)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const int HW = H * W;
    if (p >= N * HW) return;
    const int n = p / HW, rem = p - n * HW, h = rem / W, ww = rem - h * W;
    const float sn = s[n];
    float v[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        const int hh = h + t / 3 - 1, wq = ww + t % 3 - 1;
        v[t] = (hh >= 0 && hh < H && wq >= 0 && wq < W) ? x[(size_t)n * HW + hh * W + wq] / sn : 0.0f;
    }
    if (in_n) in_n[p] = v[4];
    for (int c0 = 0; c0 < C; c0 += 8) {
        u16x8 o;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int co = c0 + k;
            float a = b[co];
#pragma unroll
            for (int t = 0; t < 9; ++t) a = fmaf(w[co * 9 + t], v[t], a);
            o[k] = f2bf(fmaxf(a, 0.0f));
        }
        *reinterpret_cast<u16x8 *>(y + (size_t)p * C + c0) = o;
    }
}

// filter / bias gradient of the first convolution: dw[co][t] += sum_p g[p][co] x[p+shift(t)],
// db[co] += sum_p g[p][co], as FP32 products 16x16x4 over pixels: rows = output channels,
// columns 0..8 = the taps' shifted inputs, column 9 = ones (a thread per channel and every
// eighth pixel took 1.27 ms at 400^2 x 8).  Wave = image rows, 16 pixels per step.
__global__ __launch_bounds__(256) void k_conv_first_wgrad(const uint16_t *__restrict__ g, const float *__restrict__ x,
                                                          float *__restrict__ dw, float *__restrict__ db, int N, int H,
                                                          int W, int C)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i = lane & 15, kq = lane >> 4;
    const int co0 = blockIdx.y * 32, nw = gridDim.x * 4;
    const int dy = i / 3 - 1, dx = i % 3 - 1;
    f32x4 acc[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
    for (int row = blockIdx.x * 4 + wv; row < N * H; row += nw) {
        const int h = row % H;
        const bool rv = i < 9 && h + dy >= 0 && h + dy < H;
        const uint16_t *gr = g + (size_t)row * W * C + co0 + i;
        const float *xr = x + ((ptrdiff_t)row + dy) * W + dx;
        for (int w0 = 0; w0 < W; w0 += 16) {
            float ga[4][2], xv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int w = w0 + 4 * k + kq;
                const bool in = w < W;
                ga[k][0] = in ? bf2f(gr[(size_t)w * C]) : 0.0f;
                ga[k][1] = in ? bf2f(gr[(size_t)w * C + 16]) : 0.0f;
                xv[k] = i == 9 ? 1.0f : 0.0f;
                if (rv && in && w + dx >= 0 && w + dx < W) xv[k] = xr[w];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int f = 0; f < 2; ++f) acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(ga[k][f], xv[k], acc[f], 0, 0, 0);
        }
    }
    // lane: column i, channels 16 f + 4 kq + r
    __shared__ float red[4][2][16][16];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wv][f][4 * kq + r][i] = acc[f][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 32 * 10; e += 256) {
        const int co = e / 10, t = e - 10 * co;
        const float v = (red[0][co >> 4][co & 15][t] + red[1][co >> 4][co & 15][t]) +
                        (red[2][co >> 4][co & 15][t] + red[3][co >> 4][co & 15][t]);
        atomicAdd(t < 9 ? &dw[(co0 + co) * 9 + t] : &db[co0 + co], v);
    }
}

// relative loss: pw[b] = mean over item b of (target / s_b)^2, then the weights
// wt[b] = mean_b' pw[b'] / pw[b] (1 for an item without target power)
__global__ __launch_bounds__(1024) void k_target_power(const float *__restrict__ target, const float *__restrict__ s,
                                                      float *__restrict__ pw, int HW)
{
    const float *src = target + (size_t)blockIdx.x * HW;
    const double sb = s[blockIdx.x];
    double acc = 0.0;
    for (int i = threadIdx.x; i < HW; i += blockDim.x) {
        const double v = src[i] / sb;
        acc += v * v;
    }
    __shared__ double red[1024];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int k = blockDim.x / 2; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) pw[blockIdx.x] = (float)(red[0] / HW);
}

__global__ void k_loss_weights(float *__restrict__ wt, int B)
{
    if (threadIdx.x != 0) return;
    double m = 0.0;
    for (int b = 0; b < B; ++b) m += wt[b];
    m /= B;
    for (int b = 0; b < B; ++b) wt[b] = wt[b] > 0.0f ? (float)(m / wt[b]) : 1.0f;
}

// loss (mean squared error of the normalised output, item b weighted by wt[b] if wt) and
// head backward: d = on - target/s;  loss += wt d^2;  g_on = 2 wt d / NP;
// ga[p][ci] = g_on w[ci] (a > 0);  dw[ci] += g_on a[p][ci];  db += g_on
// Thread = 8 channels of a pixel (C / 8 neighbouring threads share one), pixels in steps of the
// grid; the channel sums meet in LDS once per workgroup (a thread per pixel with a column
// of LDS per channel took 193 us at 400^2 x 8).
__global__ __launch_bounds__(256) void k_head_loss_bwd(const uint16_t *__restrict__ a, const float *__restrict__ w,
                                                       const float *__restrict__ on, const float *__restrict__ target,
                                                       const float *__restrict__ s, const float *__restrict__ wt,
                                                       uint16_t *__restrict__ ga, float *__restrict__ dw,
                                                       float *__restrict__ db, double *__restrict__ loss, int HW, int NP,
                                                       int C)
{
    const int G = C / 8, g = threadIdx.x % G;   // G = 4 or 8
    const int step = gridDim.x * (256 / G);
    float dwl[8], wl[8], gsum = 0.0f;
    double l2 = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        dwl[k] = 0.0f;
        wl[k] = w[8 * g + k];
    }
    for (int p = blockIdx.x * (256 / G) + threadIdx.x / G; p < NP; p += step) {
        const int n = p / HW;
        const float d = on[p] - target[p] / s[n];
        const float wi = wt ? wt[n] : 1.0f;
        const float gon = 2.0f * wi * d / (float)NP;
        const u16x8 v = *reinterpret_cast<const u16x8 *>(a + (size_t)p * C + 8 * g);
        u16x8 o;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float av = bf2f(v[k]);
            o[k] = f2bf(av > 0.0f ? gon * wl[k] : 0.0f);
            dwl[k] = fmaf(gon, av, dwl[k]);
        }
        *reinterpret_cast<u16x8 *>(ga + (size_t)p * C + 8 * g) = o;
        if (g == 0) {
            gsum += gon;
            l2 += (double)(wi * d * d);
        }
    }
    l2 = block_sum_256(l2);
    if (threadIdx.x == 0) atomicAdd(loss, l2);
    __shared__ float red[256][9];
#pragma unroll
    for (int k = 0; k < 8; ++k) red[threadIdx.x][k] = dwl[k];
    red[threadIdx.x][8] = gsum;
    __syncthreads();
    if ((int)threadIdx.x <= C) {   // thread c < C: channel c, thread C: the bias
        const int c = threadIdx.x;
        float acc = 0.0f;
        for (int t = c < C ? c / 8 : 0; t < 256; t += G) acc += red[t][c < C ? c % 8 : 8];
        atomicAdd(c < C ? &dw[c] : db, acc);
    }
}

// skip-connection gradient, in place: gs[p][c] = (gs[p][c] + gp[parent(p)][c] / 4) * (act[p][c] > 0)
__global__ void k_skip_grad(uint16_t *__restrict__ gs, const uint16_t *__restrict__ act,
                            const uint16_t *__restrict__ gp, int N, int H, int W, int C)
{
    const int C8 = C / 8;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * H * W * C8) return;
    const int c8 = (int)(i % C8);
    const size_t q = i / C8;
    const int n = (int)(q / ((size_t)H * W)), rem = (int)(q - (size_t)n * H * W), h = rem / W, w = rem - h * W;
    const size_t par = ((size_t)(n * (H / 2) + h / 2) * (W / 2) + w / 2) * C + 8 * c8;
    u16x8 gv = *reinterpret_cast<const u16x8 *>(gs + q * C + 8 * c8);
    const u16x8 av = *reinterpret_cast<const u16x8 *>(act + q * C + 8 * c8);
    const u16x8 pv = *reinterpret_cast<const u16x8 *>(gp + par);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float v = bf2f(gv[k]) + 0.25f * bf2f(pv[k]);
        gv[k] = f2bf(bf2f(av[k]) > 0.0f ? v : 0.0f);
    }
    *reinterpret_cast<u16x8 *>(gs + q * C + 8 * c8) = gv;
}

// ---------------------------------------------------------------------------
// parameters: Adam, bf16 copies of the filters, flipped / transposed filters
// ---------------------------------------------------------------------------
__global__ void k_fill(float *__restrict__ p, float v, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_adam(float *__restrict__ th, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, size_t n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    th[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// wb[co][t][ci] = bf16(w[co][t][ci]);  wt[ci][t][co] = bf16(w[co][8 - t][ci])
__global__ void k_pack_filters(const float *__restrict__ w, uint16_t *__restrict__ wb, uint16_t *__restrict__ wt,
                               int Cin, int Cout)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)Cout * 9 * Cin) return;
    const int ci = (int)(i % Cin);
    const int t = (int)((i / Cin) % 9);
    const int co = (int)(i / ((size_t)9 * Cin));
    const uint16_t b = f2bf(w[i]);
    wb[i] = b;
    wt[((size_t)ci * 9 + (8 - t)) * Cout + co] = b;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct Layer {
    int cin, cout, k;         // k = 3 or 1
    size_t w_off, b_off;      // into the parameter vector
};

struct Feat {                 // one bf16 activation tensor [pixels][ch]
    uint16_t *p = nullptr;
    int ch = 0;
};

struct UNet {
    int c = 32;
    std::vector<Layer> L;     // 15 layers (see the architecture above)
    size_t nparam = 0;
    float *th = nullptr, *gr = nullptr, *m1 = nullptr, *m2 = nullptr;
    uint16_t *wb = nullptr, *wt = nullptr;
    long step = 0;
    // workspace for (B, H, W)
    int B = 0, H = 0, W = 0;
    bool grads = false;
    std::vector<void *> bufs;
    float *s = nullptr, *in_n = nullptr, *on = nullptr;
    double *sp = nullptr;  // partial sums of the image scales
    float *wpart = nullptr;   // partial filter gradients of one layer
    float *lw = nullptr;   // per-item loss weights (relative loss)
    int rel_loss = 0;      // 1: every item's squared error divided by its own normalised target power
    double *loss = nullptr;
    // s1..s3: skip connections (the concatenations themselves are never stored)
    Feat a1, s1, d1a, d1b, p1, a2, s2, d2a, d2b, p2, a3, s3, d3a, d3b, p3, a4, a4b;
    Feat g_a1, g_s1, g_d1a, g_d1b, g_p1, g_a2, g_s2, g_d2a, g_d2b, g_p2, g_a3, g_s3, g_d3a, g_d3b, g_p3, g_a4, g_a4b;
};

enum { E1A, E1B, E2A, E2B, E3A, E3B, BA, BB, D3A, D3B, D2A, D2B, D1A, D1B, HEAD, NLAYER };

static void free_ws(UNet *u)
{
    for (void *q : u->bufs) (void)hipFree(q);
    u->bufs.clear();
    u->B = u->H = u->W = 0;
    u->grads = false;
}

static int walloc(UNet *u, void **p, size_t bytes)
{
    if (device_malloc(p, std::max<size_t>(bytes, 16)) != hipSuccess) {
        (void)hipGetLastError();
        return set_error(MBREC_ERR_HIP, "mbrec:oom", "unet: device allocation of %zu bytes failed", bytes);
    }
    u->bufs.push_back(*p);
    return MBREC_OK;
}

static int feat(UNet *u, Feat &f, size_t px, int ch)
{
    f.ch = ch;
    return walloc(u, (void **)&f.p, px * ch * sizeof(uint16_t));
}

static inline unsigned nb(size_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

// splits of the pixel tiles over workgroups for the filter gradient of npair channel pairs: about
// 1024 workgroups in all (four rounds of 256 CUs' two, so that an uneven last round is small),
// a multiple of 8 (one run per XCD), and no more than there are tiles
static int wgrad_splits(int npair, int ntiles)
{
    const int want = std::max(8, (1024 / npair + 7) / 8 * 8);
    return std::min(want, std::max(1, ntiles));
}

// columns of the virtual wide image, and its tiles of `rows` rows
struct ConvGrid {
    int Wp, tiles_x, ntiles;
    ConvGrid(int N, int H, int W, int rows)
        : Wp(W + (W % 2 ? 1 : 2)), tiles_x((int)(((size_t)N * Wp + kCvCols - 1) / kCvCols)),
          ntiles(tiles_x * ((H + rows - 1) / rows)) {}
};

static int ensure_ws(UNet *u, int B, int H, int W, bool grads)
{
    if (u->B == B && u->H == H && u->W == W && (u->grads || !grads)) return MBREC_OK;
    MBREC_HIP(hipDeviceSynchronize());
    free_ws(u);
    const int c = u->c;
    const size_t P1 = (size_t)B * H * W, P2 = P1 / 4, P3 = P1 / 16, P4 = P1 / 64;
    int rc;
    if ((rc = walloc(u, (void **)&u->s, sizeof(float) * B)) || (rc = walloc(u, (void **)&u->lw, sizeof(float) * B)) ||
        (rc = walloc(u, (void **)&u->sp, sizeof(double) * B * kScaleParts)) ||
        (rc = walloc(u, (void **)&u->loss, sizeof(double))) ||
        (rc = feat(u, u->a1, P1, c)) || (rc = feat(u, u->s1, P1, c)) || (rc = feat(u, u->d1a, P1, c)) ||
        (rc = feat(u, u->p1, P2, c)) || (rc = feat(u, u->a2, P2, 2 * c)) ||
        (rc = feat(u, u->s2, P2, 2 * c)) || (rc = feat(u, u->d2a, P2, 2 * c)) || (rc = feat(u, u->d2b, P2, 2 * c)) ||
        (rc = feat(u, u->p2, P3, 2 * c)) || (rc = feat(u, u->a3, P3, 4 * c)) || (rc = feat(u, u->s3, P3, 4 * c)) ||
        (rc = feat(u, u->d3a, P3, 4 * c)) || (rc = feat(u, u->d3b, P3, 4 * c)) || (rc = feat(u, u->p3, P4, 4 * c)) ||
        (rc = feat(u, u->a4, P4, 8 * c)) || (rc = feat(u, u->a4b, P4, 8 * c))) {
        free_ws(u);
        return rc;
    }
    u->in_n = u->on = nullptr;
    u->d1b = Feat{nullptr, c};
    if (grads) {
        size_t part = 0;
        for (int l = E1B; l <= D1B; ++l) {
            const int lev = l <= E1B ? 0 : l <= E2B ? 1 : l <= E3B ? 2 : l <= BB ? 3 : l <= D3B ? 2 : l <= D2B ? 1 : 0;
            const int npair = (u->L[l].cin / 32) * (u->L[l].cout / 32);
            part = std::max(part, (size_t)npair * wgrad_splits(npair, ConvGrid(B, H >> lev, W >> lev, kWgRows).ntiles));
        }
        if ((rc = walloc(u, (void **)&u->in_n, sizeof(float) * P1)) ||
            (rc = walloc(u, (void **)&u->on, sizeof(float) * P1)) || (rc = feat(u, u->d1b, P1, c)) ||
            (rc = walloc(u, (void **)&u->wpart, sizeof(float) * part * kWgPart)) ||
            (rc = feat(u, u->g_a1, P1, c)) || (rc = feat(u, u->g_s1, P1, c)) || (rc = feat(u, u->g_d1a, P1, c)) ||
            (rc = feat(u, u->g_d1b, P1, c)) || (rc = feat(u, u->g_p1, P2, c)) || (rc = feat(u, u->g_a2, P2, 2 * c)) ||
            (rc = feat(u, u->g_s2, P2, 2 * c)) || (rc = feat(u, u->g_d2a, P2, 2 * c)) ||
            (rc = feat(u, u->g_d2b, P2, 2 * c)) || (rc = feat(u, u->g_p2, P3, 2 * c)) ||
            (rc = feat(u, u->g_a3, P3, 4 * c)) || (rc = feat(u, u->g_s3, P3, 4 * c)) ||
            (rc = feat(u, u->g_d3a, P3, 4 * c)) || (rc = feat(u, u->g_d3b, P3, 4 * c)) ||
            (rc = feat(u, u->g_p3, P4, 4 * c)) || (rc = feat(u, u->g_a4, P4, 8 * c)) ||
            (rc = feat(u, u->g_a4b, P4, 8 * c))) {
            free_ws(u);
            return rc;
        }
    }
    u->B = B;
    u->H = H;
    u->W = W;
    u->grads = grads;
    return MBREC_OK;
}

static ConvSrc whole(const Feat &f) { return ConvSrc{f.p, f.ch, 0, 0}; }
static ConvSrc upsampled(const Feat &f) { return ConvSrc{f.p, f.ch, 0, 1}; }

// common arguments of a convolution over x (one source), cin -> cout at N x H x W
static ConvArgs conv_args(const ConvSrc &x, int cin, const uint16_t *w, int cout, int N, int H, int W)
{
    ConvArgs a{};
    a.src[0] = a.src[1] = x;
    a.split = a.Cin = cin;
    a.Cout = cout;
    a.w = w;
    a.N = N;
    a.H = H;
    a.W = W;
    const ConvGrid g(N, H, W, kCvRows);
    a.Wp = g.Wp;
    a.tiles_x = g.tiles_x;
    a.ntiles = g.ntiles;
    return a;
}

template <int NB, int EPI, typename T>
static void conv_run(ConvArgs &a, hipStream_t s)
{
    a.ncot = a.Cout / (32 * NB);
    // a launch holds fewer than 2^32 threads: 2^23 workgroups at most, in whole runs of eight tiles
    const int run = std::max(8, (1 << 23) / a.ncot / 8 * 8);
    for (a.tile0 = 0; a.tile0 < a.ntiles; a.tile0 += run) {
        const dim3 grid((unsigned)((std::min(run, a.ntiles - a.tile0) + 7) / 8 * 8 * (size_t)a.ncot));
        hipLaunchKernelGGL((k_conv3<NB, EPI, T>), grid, dim3(256), 0, s, a);
    }
}

// 32 output channels per workgroup; 64 where the head reads as many, and for long sums (192 input channels and
// more) in launches that fill the chip many times over, where reading the pixels half as often counts: the network
// of base width 64 on 32 images of 400^2 8.0 ms against 8.25 (tiles of 16 rows: 7.8), that of 32 on 64 images 5.2 ms either way
// (64 channels for every layer that divides: 5.4).
template <int EPI, typename T = int>
static void conv_launch(ConvArgs &a, hipStream_t s)
{
    const bool wide = EPI == kHead ? a.Cout == 64
                                   : a.Cout % 64 == 0 && a.Cin >= 192 && (size_t)a.ntiles * (a.Cout / 64) >= 4096;
    wide ? conv_run<2, EPI, T>(a, s) : conv_run<1, EPI, T>(a, s);
}

// y = relu(conv3x3(x) + bias); pool (may be null): also its 2 x 2 average
static void conv_relu(const ConvSrc &x, int cin, const uint16_t *w, const float *bias, const Feat &y, const Feat *pool,
                      int N, int H, int W, hipStream_t s)
{
    ConvArgs a = conv_args(x, cin, w, y.ch, N, H, W);
    a.bias = bias;
    a.y = y.p;
    a.ys = y.ch;
    a.yp = pool ? pool->p : nullptr;
    conv_launch<kRelu>(a, s);
}

// the same over the concatenation (upsampled low, skip)
static void conv_cat(const Feat &low, const Feat &skip, const uint16_t *w, const float *bias, const Feat &y, int N, int H,
                     int W, hipStream_t s)
{
    ConvArgs a = conv_args(upsampled(low), low.ch, w, y.ch, N, H, W);
    a.src[1] = whole(skip);
    a.Cin = low.ch + skip.ch;
    a.bias = bias;
    a.y = y.p;
    a.ys = y.ch;
    conv_launch<kRelu>(a, s);
}

// input gradient: y = conv3x3(g) with the flipped filters, where mask (may be null) > 0
static void conv_grad(const Feat &g, const uint16_t *w, const Feat &y, const Feat *mask, int N, int H, int W,
                      hipStream_t s)
{
    ConvArgs a = conv_args(whole(g), g.ch, w, y.ch, N, H, W);
    a.y = y.p;
    a.ys = y.ch;
    a.m = mask ? mask->p : nullptr;
    a.ms = mask ? mask->ch : 0;
    conv_launch<kGrad>(a, s);
}

// input gradient of a concatenation: g_low (through the upsampling, where low > 0) and g_skip
static void conv_grad_cat(const Feat &g, const uint16_t *w, const Feat &g_low, const Feat &low, const Feat &g_skip, int N,
                          int H, int W, hipStream_t s)
{
    ConvArgs a = conv_args(whole(g), g.ch, w, low.ch + g_skip.ch, N, H, W);
    a.y = g_skip.p;
    a.ys = g_skip.ch;
    a.yp = g_low.p;
    a.mp = low.p;
    a.n_low = low.ch;
    conv_launch<kGradUp>(a, s);
}

// dw, db of the convolution of x (x2: the second part of a concatenation, x then at half resolution)
static void wgrad3(UNet *u, const Feat &g, const Feat &x, const Feat *x2, float *dw, float *db, int N, int H, int W,
                   hipStream_t s)
{
    const ConvGrid cg(N, H, W, kWgRows);
    WgradArgs a{};
    a.g = whole(g);
    a.src[0] = x2 ? upsampled(x) : whole(x);
    a.src[1] = x2 ? whole(*x2) : a.src[0];
    a.split = x.ch;
    a.Cin = x.ch + (x2 ? x2->ch : 0);
    a.Cout = g.ch;
    a.part = u->wpart;
    a.N = N;
    a.H = H;
    a.W = W;
    a.Wp = cg.Wp;
    a.tiles_x = cg.tiles_x;
    a.ntiles = cg.ntiles;
    a.npair = (a.Cin / 32) * (a.Cout / 32);
    a.nsplit = wgrad_splits(a.npair, a.ntiles);
    const unsigned grid = (unsigned)((a.nsplit + 7) / 8 * 8 * a.npair);
    hipLaunchKernelGGL(k_conv3_wgrad, dim3(grid), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_wgrad_sum, dim3(289, a.npair), dim3(256), 0, s, (const float *)u->wpart, dw, db, a.Cin, a.nsplit);
}

static void pack_all(UNet *u, hipStream_t s)
{
    for (int l = E1B; l <= D1B; ++l) {
        const Layer &ly = u->L[l];
        const size_t n = (size_t)ly.cout * 9 * ly.cin;
        hipLaunchKernelGGL(k_pack_filters, dim3(nb(n)), dim3(256), 0, s, u->th + ly.w_off, u->wb + ly.w_off,
                           u->wt + ly.w_off, ly.cin, ly.cout);
    }
}

static const uint16_t *WB(UNet *u, int l) { return u->wb + u->L[l].w_off; }
static const uint16_t *WT(UNet *u, int l) { return u->wt + u->L[l].w_off; }
static const float *BIAS(UNet *u, int l) { return u->th + u->L[l].b_off; }

// the network on `in`; grads: keep what the backward pass reads
static int forward(UNet *u, const float *in, float *out, int B, int H, int W, bool grads, hipStream_t s)
{
    const int c = u->c;
    const int HW = H * W;
    const size_t P1 = (size_t)B * HW;
    hipLaunchKernelGGL(k_image_sumsq, dim3(kScaleParts, B), dim3(256), 0, s, in, u->sp, HW);
    hipLaunchKernelGGL(k_image_scale, dim3(nb(B, 64)), dim3(64), 0, s, (const double *)u->sp, u->s, B, HW);
    hipLaunchKernelGGL(k_conv_first, dim3(nb(P1)), dim3(256), 0, s, in, (const float *)u->s, grads ? u->in_n : nullptr,
                       u->th + u->L[E1A].w_off, BIAS(u, E1A), u->a1.p, B, H, W, c);
    const int H2 = H / 2, W2 = W / 2, H3 = H / 4, W3 = W / 4, H4 = H / 8, W4 = W / 8;
    auto conv = [&](const Feat &x, int l, const Feat &y, const Feat *pool, int h, int w) {
        conv_relu(whole(x), x.ch, WB(u, l), BIAS(u, l), y, pool, B, h, w, s);
    };
    // encoder
    conv(u->a1, E1B, u->s1, &u->p1, H, W);
    conv(u->p1, E2A, u->a2, nullptr, H2, W2);
    conv(u->a2, E2B, u->s2, &u->p2, H2, W2);
    conv(u->p2, E3A, u->a3, nullptr, H3, W3);
    conv(u->a3, E3B, u->s3, &u->p3, H3, W3);
    conv(u->p3, BA, u->a4, nullptr, H4, W4);
    conv(u->a4, BB, u->a4b, nullptr, H4, W4);
    // decoder
    conv_cat(u->a4b, u->s3, WB(u, D3A), BIAS(u, D3A), u->d3a, B, H3, W3, s);
    conv(u->d3a, D3B, u->d3b, nullptr, H3, W3);
    conv_cat(u->d3b, u->s2, WB(u, D2A), BIAS(u, D2A), u->d2a, B, H2, W2, s);
    conv(u->d2a, D2B, u->d2b, nullptr, H2, W2);
    conv_cat(u->d2b, u->s1, WB(u, D1A), BIAS(u, D1A), u->d1a, B, H, W, s);
    // last convolution with the head (all c channels are one workgroup's)
    ConvArgs a = conv_args(whole(u->d1a), c, WB(u, D1B), c, B, H, W);
    a.bias = BIAS(u, D1B);
    a.y = grads ? u->d1b.p : nullptr;
    a.ys = c;
    a.hw = u->th + u->L[HEAD].w_off;
    a.hb = BIAS(u, HEAD);
    a.s = u->s;
    a.on = grads ? u->on : nullptr;
    a.out = out;
    conv_launch<kHead>(a, s);
    MBREC_HIP(hipGetLastError());
    return MBREC_OK;
}

static float *GW(UNet *u, int l) { return u->gr + u->L[l].w_off; }
static float *GB(UNet *u, int l) { return u->gr + u->L[l].b_off; }

// gradients of the loss with respect to all parameters (u->gr, zeroed here)
static int backward(UNet *u, const float *target, int B, int H, int W, hipStream_t s)
{
    const int c = u->c;
    const int HW = H * W;
    const size_t P1 = (size_t)B * HW;
    const int H2 = H / 2, W2 = W / 2, H3 = H / 4, W3 = W / 4, H4 = H / 8, W4 = W / 8;
    hipLaunchKernelGGL(k_fill, dim3(nb(u->nparam)), dim3(256), 0, s, u->gr, 0.0f, u->nparam);
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(64), 0, s, (float *)u->loss, 0.0f, (size_t)2);
    if (u->rel_loss) {
        hipLaunchKernelGGL(k_target_power, dim3(B), dim3(1024), 0, s, target, (const float *)u->s, u->lw, HW);
        hipLaunchKernelGGL(k_loss_weights, dim3(1), dim3(64), 0, s, u->lw, B);
    }
    hipLaunchKernelGGL(k_head_loss_bwd, dim3(std::min(2048u, nb(P1, 2048 / c))), dim3(256), 0, s, u->d1b.p,
                       u->th + u->L[HEAD].w_off, u->on,
                       target, u->s, u->rel_loss ? (const float *)u->lw : nullptr, u->g_d1b.p, GW(u, HEAD),
                       GB(u, HEAD), u->loss, HW, (int)P1, c);
    auto layer = [&](int l, const Feat &g, const Feat &x, const Feat &gx, const Feat *mask, int h, int w) {
        wgrad3(u, g, x, nullptr, GW(u, l), GB(u, l), B, h, w, s);
        conv_grad(g, WT(u, l), gx, mask, B, h, w, s);
    };
    auto layer_cat = [&](int l, const Feat &g, const Feat &low, const Feat &skip, const Feat &g_low, const Feat &g_skip,
                         int h, int w) {
        wgrad3(u, g, low, &skip, GW(u, l), GB(u, l), B, h, w, s);
        conv_grad_cat(g, WT(u, l), g_low, low, g_skip, B, h, w, s);
    };
    auto skip = [&](const Feat &g, const Feat &act, const Feat &gp, int h, int w) {
        hipLaunchKernelGGL(k_skip_grad, dim3(nb((size_t)B * h * w * g.ch / 8)), dim3(256), 0, s, g.p, act.p, gp.p, B, h,
                           w, g.ch);
    };
    layer(D1B, u->g_d1b, u->d1a, u->g_d1a, &u->d1a, H, W);
    layer_cat(D1A, u->g_d1a, u->d2b, u->s1, u->g_d2b, u->g_s1, H, W);
    layer(D2B, u->g_d2b, u->d2a, u->g_d2a, &u->d2a, H2, W2);
    layer_cat(D2A, u->g_d2a, u->d3b, u->s2, u->g_d3b, u->g_s2, H2, W2);
    layer(D3B, u->g_d3b, u->d3a, u->g_d3a, &u->d3a, H3, W3);
    layer_cat(D3A, u->g_d3a, u->a4b, u->s3, u->g_a4b, u->g_s3, H3, W3);
    layer(BB, u->g_a4b, u->a4, u->g_a4, &u->a4, H4, W4);
    layer(BA, u->g_a4, u->p3, u->g_p3, nullptr, H4, W4);
    skip(u->g_s3, u->s3, u->g_p3, H3, W3);
    layer(E3B, u->g_s3, u->a3, u->g_a3, &u->a3, H3, W3);
    layer(E3A, u->g_a3, u->p2, u->g_p2, nullptr, H3, W3);
    skip(u->g_s2, u->s2, u->g_p2, H2, W2);
    layer(E2B, u->g_s2, u->a2, u->g_a2, &u->a2, H2, W2);
    layer(E2A, u->g_a2, u->p1, u->g_p1, nullptr, H2, W2);
    skip(u->g_s1, u->s1, u->g_p1, H, W);
    layer(E1B, u->g_s1, u->a1, u->g_a1, &u->a1, H, W);
    hipLaunchKernelGGL(k_conv_first_wgrad, dim3(std::min(512u, nb((size_t)B * H, 4)), c / 32), dim3(256), 0, s, u->g_a1.p,
                       u->in_n, GW(u, E1A), GB(u, E1A), B, H, W, c);
    MBREC_HIP(hipGetLastError());
    return MBREC_OK;
}

static int check_shape(UNet *u, int B, int H, int W)
{
    if (B <= 0 || H <= 0 || W <= 0 || H % 8 || W % 8)
        return set_error(MBREC_ERR_ARG, "mbrec:unetShape", "unet: B, H, W must be positive and H, W multiples of 8 "
                                                           "(got B=%d H=%d W=%d)", B, H, W);
    if ((size_t)B * H * W * 12 * u->c > (size_t)INT32_MAX * 4)
        return set_error(MBREC_ERR_ARG, "mbrec:unetShape", "unet: batch too large");
    return MBREC_OK;
}

}  // namespace mbrec

using namespace mbrec;

struct mbrec_unet_s {
    UNet u;
};

extern "C" {

int mbrec_unet_create(mbrec_unet *out, int base_channels, unsigned long long seed)
{
    if (!out) return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_create: null output");
    *out = nullptr;
    if (base_channels <= 0 || base_channels % 32 || base_channels > 64)
        return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_create: base_channels must be 32 or 64 (got %d)",
                         base_channels);
    mbrec_unet h = new mbrec_unet_s;
    UNet *u = &h->u;
    const int c = base_channels;
    u->c = c;
    const int io[NLAYER][3] = {{1, c, 3},          {c, c, 3},          {c, 2 * c, 3},      {2 * c, 2 * c, 3},
                               {2 * c, 4 * c, 3},  {4 * c, 4 * c, 3},  {4 * c, 8 * c, 3},  {8 * c, 8 * c, 3},
                               {12 * c, 4 * c, 3}, {4 * c, 4 * c, 3},  {6 * c, 2 * c, 3},  {2 * c, 2 * c, 3},
                               {3 * c, c, 3},      {c, c, 3},          {c, 1, 1}};
    size_t off = 0;
    for (int l = 0; l < NLAYER; ++l) {
        Layer ly{io[l][0], io[l][1], io[l][2], 0, 0};
        ly.w_off = off;
        off += (size_t)ly.cout * ly.k * ly.k * ly.cin;
        ly.b_off = off;
        off += (size_t)ly.cout;
        off = (off + 7) / 8 * 8;   // keep every filter 16-byte aligned in the bf16 copies
        u->L.push_back(ly);
    }
    u->nparam = off;
    // He-normal filters, zero biases (seeded splitmix64 + Box-Muller)
    std::vector<float> th(off, 0.0f);
    uint64_t st = seed ^ 0x9e3779b97f4a7c15ull;
    auto next = [&]() {
        uint64_t z = (st += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        z ^= z >> 31;
        return ((z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    for (int l = 0; l < NLAYER; ++l) {
        const Layer &ly = u->L[l];
        const size_t n = (size_t)ly.cout * ly.k * ly.k * ly.cin;
        const double sd = std::sqrt(2.0 / (ly.k * ly.k * ly.cin)) * (l == HEAD ? 0.5 : 1.0);
        for (size_t i = 0; i < n; ++i) {
            const double u1 = next(), u2 = next();
            th[ly.w_off + i] = (float)(sd * std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2));
        }
    }
    auto fail = [&](int rc) {
        mbrec_unet_destroy(h);
        return rc;
    };
    const size_t bytes = sizeof(float) * off;
    if (hipMalloc((void **)&u->th, bytes) != hipSuccess || hipMalloc((void **)&u->gr, bytes) != hipSuccess ||
        hipMalloc((void **)&u->m1, bytes) != hipSuccess || hipMalloc((void **)&u->m2, bytes) != hipSuccess ||
        hipMalloc((void **)&u->wb, sizeof(uint16_t) * off) != hipSuccess ||
        hipMalloc((void **)&u->wt, sizeof(uint16_t) * off) != hipSuccess) {
        (void)hipGetLastError();
        return fail(set_error(MBREC_ERR_HIP, "mbrec:oom", "unet_create: device allocation failed"));
    }
    if (hipMemcpy(u->th, th.data(), bytes, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(u->m1, 0, bytes) != hipSuccess || hipMemset(u->m2, 0, bytes) != hipSuccess ||
        hipMemset(u->gr, 0, bytes) != hipSuccess || hipMemset(u->wb, 0, sizeof(uint16_t) * off) != hipSuccess ||
        hipMemset(u->wt, 0, sizeof(uint16_t) * off) != hipSuccess)
        return fail(set_error(MBREC_ERR_HIP, "mbrec:hip", "unet_create: upload failed"));
    pack_all(u, 0);
    if (hipDeviceSynchronize() != hipSuccess) return fail(set_error(MBREC_ERR_HIP, "mbrec:hip", "unet_create: pack"));
    *out = h;
    return MBREC_OK;
}

int mbrec_unet_destroy(mbrec_unet h)
{
    if (!h) return MBREC_OK;
    (void)hipDeviceSynchronize();
    UNet *u = &h->u;
    free_ws(u);
    void *p[] = {u->th, u->gr, u->m1, u->m2, u->wb, u->wt};
    for (void *q : p)
        if (q) (void)hipFree(q);
    delete h;
    return MBREC_OK;
}

size_t mbrec_unet_num_params(mbrec_unet h) { return h ? h->u.nparam : 0; }

int mbrec_unet_layout(mbrec_unet h, int layer, int *cin, int *cout, int *ksize, size_t *w_off, size_t *b_off)
{
    if (!h || layer < 0 || layer >= NLAYER) return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_layout: bad layer");
    const Layer &ly = h->u.L[layer];
    *cin = ly.cin;
    *cout = ly.cout;
    *ksize = ly.k;
    *w_off = ly.w_off;
    *b_off = ly.b_off;
    return MBREC_OK;
}

int mbrec_unet_get_params(mbrec_unet h, float *host, size_t n)
{
    if (!h || !host || n != h->u.nparam)
        return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_get_params: expected %zu values", h ? h->u.nparam : 0);
    MBREC_HIP(hipDeviceSynchronize());
    MBREC_HIP(hipMemcpy(host, h->u.th, sizeof(float) * n, hipMemcpyDeviceToHost));
    return MBREC_OK;
}

int mbrec_unet_set_params(mbrec_unet h, const float *host, size_t n)
{
    if (!h || !host || n != h->u.nparam)
        return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_set_params: expected %zu values", h ? h->u.nparam : 0);
    UNet *u = &h->u;
    MBREC_HIP(hipDeviceSynchronize());
    MBREC_HIP(hipMemcpy(u->th, host, sizeof(float) * n, hipMemcpyHostToDevice));
    MBREC_HIP(hipMemset(u->m1, 0, sizeof(float) * n));
    MBREC_HIP(hipMemset(u->m2, 0, sizeof(float) * n));
    u->step = 0;
    pack_all(u, 0);
    MBREC_HIP(hipDeviceSynchronize());
    return MBREC_OK;
}

int mbrec_unet_forward(mbrec_unet h, const float *in, float *out, int B, int H, int W, mbrec_stream stream)
{
    if (!h || !in || !out) return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_forward: null argument");
    UNet *u = &h->u;
    int rc;
    if ((rc = check_shape(u, B, H, W))) return rc;
    if ((rc = ensure_ws(u, B, H, W, false))) return rc;
    return forward(u, in, out, B, H, W, false, (hipStream_t)stream);
}

int mbrec_unet_gradients(mbrec_unet h, const float *in, const float *target, int B, int H, int W, float *grad_host,
                         double *loss_host, mbrec_stream stream)
{
    if (!h || !in || !target) return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_gradients: null argument");
    UNet *u = &h->u;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if ((rc = check_shape(u, B, H, W))) return rc;
    if ((rc = ensure_ws(u, B, H, W, true))) return rc;
    if ((rc = forward(u, in, nullptr, B, H, W, true, s))) return rc;
    if ((rc = backward(u, target, B, H, W, s))) return rc;
    MBREC_HIP(hipStreamSynchronize(s));
    if (grad_host) MBREC_HIP(hipMemcpy(grad_host, u->gr, sizeof(float) * u->nparam, hipMemcpyDeviceToHost));
    if (loss_host) {
        double l = 0.0;
        MBREC_HIP(hipMemcpy(&l, u->loss, sizeof(double), hipMemcpyDeviceToHost));
        *loss_host = l / ((double)B * H * W);
    }
    return MBREC_OK;
}

int mbrec_unet_set_relative_loss(mbrec_unet h, int on)
{
    if (!h) return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_set_relative_loss: null argument");
    h->u.rel_loss = on ? 1 : 0;
    return MBREC_OK;
}

int mbrec_unet_train_step(mbrec_unet h, const float *in, const float *target, int B, int H, int W, float lr,
                          float beta1, float beta2, float eps, double *loss_host, mbrec_stream stream)
{
    if (!h || !in || !target) return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_train_step: null argument");
    if (!(lr > 0.0f) || !(beta1 >= 0.0f && beta1 < 1.0f) || !(beta2 >= 0.0f && beta2 < 1.0f) || !(eps > 0.0f))
        return set_error(MBREC_ERR_ARG, "mbrec:args", "unet_train_step: invalid Adam settings");
    UNet *u = &h->u;
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if ((rc = check_shape(u, B, H, W))) return rc;
    if ((rc = ensure_ws(u, B, H, W, true))) return rc;
    if ((rc = forward(u, in, nullptr, B, H, W, true, s))) return rc;
    if ((rc = backward(u, target, B, H, W, s))) return rc;
    ++u->step;
    const float c1 = 1.0f - std::pow(beta1, (float)u->step), c2 = 1.0f - std::pow(beta2, (float)u->step);
    hipLaunchKernelGGL(k_adam, dim3(nb(u->nparam)), dim3(256), 0, s, u->th, u->gr, u->m1, u->m2, u->nparam, lr, beta1,
                       beta2, eps, c1, c2);
    pack_all(u, s);
    MBREC_HIP(hipGetLastError());
    if (loss_host) {
        double l = 0.0;
        MBREC_HIP(hipMemcpyAsync(&l, u->loss, sizeof(double), hipMemcpyDeviceToHost, s));
        MBREC_HIP(hipStreamSynchronize(s));
        *loss_host = l / ((double)B * H * W);
    }
    return MBREC_OK;
}

// One 3x3 convolution layer (bf16 NHWC input [N][H][W][Cin], bf16 filters
// [Cout][3][3][Cin], FP32 bias, + ReLU) through the matrix-core kernel.
int mbrec_conv3x3_bf16(const uint16_t *x, const uint16_t *w, const float *bias, uint16_t *y, int N, int H, int W,
                       int Cin, int Cout, int relu, mbrec_stream stream)
{
    if (!x || !w || !y || N <= 0 || H <= 0 || W <= 0 || Cin % 32 || Cout % 32 || Cin <= 0 || Cout <= 0)
        return set_error(MBREC_ERR_ARG, "mbrec:args", "conv3x3_bf16: Cin and Cout must be positive multiples of 32");
    // pixel and virtual column indices (at most two columns a pixel, one tile past the end) are 32-bit
    constexpr size_t lim = ((size_t)1 << 30) - 64;
    if ((size_t)N * H >= lim || (size_t)N * H * W >= lim)
        return set_error(MBREC_ERR_ARG, "mbrec:args", "conv3x3_bf16: N * H * W must be below 2^30 - 64");
    // the kernel reads and writes 16- and 8-byte pieces: arrays at other addresses go through aligned copies
    hipStream_t s = (hipStream_t)stream;
    if (!relu && bias) return set_error(MBREC_ERR_ARG, "mbrec:args", "conv3x3_bf16: bias requires relu=1");
    const size_t nx = (size_t)N * H * W * Cin * 2, nw = (size_t)Cout * 9 * Cin * 2, ny = (size_t)N * H * W * Cout * 2;
    struct Copies {
        hipStream_t s;
        void *x = nullptr, *w = nullptr, *y = nullptr;
        ~Copies()
        {
            for (void *q : {x, w, y})
                if (q) (void)hipFreeAsync(q, s);
        }
    } c{s};
    if ((uintptr_t)x % 16) {
        MBREC_HIP(hipMallocAsync(&c.x, nx, s));
        MBREC_HIP(hipMemcpyAsync(c.x, x, nx, hipMemcpyDeviceToDevice, s));
    }
    if ((uintptr_t)w % 16) {
        MBREC_HIP(hipMallocAsync(&c.w, nw, s));
        MBREC_HIP(hipMemcpyAsync(c.w, w, nw, hipMemcpyDeviceToDevice, s));
    }
    if ((uintptr_t)y % 8) MBREC_HIP(hipMallocAsync(&c.y, ny, s));
    const Feat fx{c.x ? (uint16_t *)c.x : const_cast<uint16_t *>(x), Cin}, fy{c.y ? (uint16_t *)c.y : y, Cout};
    const uint16_t *fw = c.w ? (const uint16_t *)c.w : w;
    ConvArgs a = conv_args(whole(fx), Cin, fw, Cout, N, H, W);
    a.y = fy.p;
    a.ys = Cout;
    a.bias = bias;
    const bool far = nx / 16 >= (size_t)INT32_MAX;   // slots beyond 32-bit indices
    if (relu) far ? conv_launch<kRelu, long long>(a, s) : conv_launch<kRelu>(a, s);
    else far ? conv_launch<kGrad, long long>(a, s) : conv_launch<kGrad>(a, s);   // plain convolution
    MBREC_HIP(hipGetLastError());
    if (c.y) MBREC_HIP(hipMemcpyAsync(y, c.y, ny, hipMemcpyDeviceToDevice, s));
    return MBREC_OK;
}

}  // extern "C"
