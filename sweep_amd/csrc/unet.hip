// Kernels of the learned preconditioner: bfloat16 convolutions on the
// matrix cores (v_mfma_f32_16x16x32_bf16, float32 accumulation) and the
// element-wise passes of a 2-D U-Net's forward and backward.
//
// The convolution is an implicit GEMM over NHWC views: D[pixel, co] =
// sum_k A[pixel, k] B[k, co] with k = (tap, ci).  A 16 x 16 x 32 MFMA takes,
// in lane l, row l % 16 of A and column l % 16 of B, each with 8 of the 32
// k values (the same 8 in both, lane group l / 16 holding k = 8 (l / 16) ..
// + 7 here), and returns D[4 (l / 16) + e][l % 16] in element e.  With
// cin a multiple of 8 a lane's 8 k values are 8 consecutive channels of one
// tap: one 16-byte load from the NHWC input and one from the weights.
//
// The weight gradient reduces over pixels, which are not contiguous in
// either operand; its transposing LDS reads are described at its kernel.  The
// pixel range is split across workgroups and the float32 partial tiles are
// summed in a fixed order by a second kernel.
#include "unet.h"

#include <algorithm>
#include <cmath>

namespace swp {
namespace nn {

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;

__device__ __forceinline__ float bf2f(uint16_t h) { return __builtin_bit_cast(float, uint32_t(h) << 16); }

__device__ __forceinline__ uint16_t f2bf(float f)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40u);
    return uint16_t((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ bf16x8 ld8(const uint16_t *p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p));
}

__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u}); }

__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------- forward
// At most 32 input channels (one MFMA step a tap).  Block: 4 waves, 64 columns x
// 4 rows of pixels (a row a wave) x 16 NT output channels.  The block stages its
// pixels with their halo in LDS once for all taps, and the weights a row of taps
// at a time; a wave's 4 x NT MFMAs of a tap then take 4 + NT fragments from LDS (16
// bytes a lane, rows of 80 bytes: the 16 lanes of a group on 16 different bank
// quads).  The weights are the first operand, so a lane ends up with four
// consecutive channels of a pixel and stores them together.  The next phase's
// global loads are in flight while a phase multiplies.
// NT 4 from 33 channels up, 2 from 17, else 1: the network's 32- and 8-channel
// layers multiplied 2 and 8 times their channels in tiles of 64.  Measured in a
// 2 x 384 x 1152, base-32 training step: 32 -> 32 about 110 -> 43 us.
constexpr int kCPitch = 40;   // LDS row (32 channels of a pixel or weight row) in halves

template <int KS, int NT, bool F32OUT>
__global__ void __launch_bounds__(256, 2) conv_c32_kernel(const uint16_t *__restrict__ in, int H, int W, int cin,
                                                          int is, const uint16_t *__restrict__ w, int cout,
                                                          const float *__restrict__ bias, int relu,
                                                          void *__restrict__ out, int os, int ncot, int vec)
{
    constexpr int R = KS / 2, IW = 64 + 2 * R, IH = 4 + 2 * R, CO = 16 * NT;
    constexpr int UI = (IH * IW * 4 + 255) / 256, UW = (KS * CO * 4 + 255) / 256;   // 16-byte units a thread
    __shared__ __attribute__((aligned(16))) uint16_t sI[IH * IW * kCPitch];
    __shared__ __attribute__((aligned(16))) uint16_t sW[KS * CO * kCPitch];
    const int tid = int(threadIdx.x), lane = tid & 63, wv = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int x0 = int(blockIdx.x) * 64, y0 = int(blockIdx.y) * 4;
    const int n = int(blockIdx.z) / ncot, co0 = (int(blockIdx.z) % ncot) * CO;
    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 ri[UI], rw[UW];
    auto fetch_in = [&] {   // the pixels and their halo (zeros outside)
#pragma unroll
        for (int u = 0; u < UI; ++u) {
            const int k = tid + 256 * u, px = k >> 2, ci = (k & 3) * 8;
            const int y = y0 - R + px / IW, x = x0 - R + px % IW;
            ri[u] = u32x4{0u, 0u, 0u, 0u};
            if (px < IH * IW && ci < cin && y >= 0 && y < H && x >= 0 && x < W)
                ri[u] = *reinterpret_cast<const u32x4 *>(in + ((int64_t(n) * H + y) * W + x) * is + ci);
        }
    };
    auto fetch_w = [&](int dy) {   // the KS taps of row dy
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            const int k = tid + 256 * u, row = k >> 2, ci = (k & 3) * 8;
            const int dx = row / CO, co = co0 + row % CO;
            rw[u] = u32x4{0u, 0u, 0u, 0u};
            if (row < KS * CO && ci < cin && co < cout)
                rw[u] = *reinterpret_cast<const u32x4 *>(w + (int64_t(co) * (KS * KS) + dy * KS + dx) * cin + ci);
        }
    };
    fetch_in();
    fetch_w(0);
#pragma unroll
    for (int dy = 0; dy < KS; ++dy) {
        __syncthreads();
        if (dy == 0) {
#pragma unroll
            for (int u = 0; u < UI; ++u) {
                const int k = tid + 256 * u;
                if (k < IH * IW * 4) *reinterpret_cast<u32x4 *>(sI + (k >> 2) * kCPitch + (k & 3) * 8) = ri[u];
            }
        }
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            const int k = tid + 256 * u;
            if (k < KS * CO * 4) *reinterpret_cast<u32x4 *>(sW + (k >> 2) * kCPitch + (k & 3) * 8) = rw[u];
        }
        __syncthreads();
        if (dy + 1 < KS) fetch_w(dy + 1);
#pragma unroll
        for (int dx = 0; dx < KS; ++dx) {
            bf16x8 wf[NT], px[4];
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[t] = ld8(sW + (dx * CO + 16 * t + r16) * kCPitch + 8 * g);
#pragma unroll
            for (int m = 0; m < 4; ++m) px[m] = ld8(sI + ((wv + dy) * IW + 16 * m + r16 + dx) * kCPitch + 8 * g);
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[m][t] = mma(wf[t], px[m], acc[m][t]);
        }
    }
    const int y = y0 + wv;
    if (y >= H) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + 16 * t + 4 * g;
        if (co >= cout) continue;
        float bv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[e] = bias && co + e < cout ? bias[co + e] : 0.f;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int x = x0 + 16 * m + r16;
            if (x >= W) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = acc[m][t][e] + bv[e];
                if (relu) v[e] = fmaxf(v[e], 0.f);
            }
            const int64_t i = ((int64_t(n) * H + y) * W + x) * os + co;
            if (vec && co + 4 <= cout) {   // four channels in one store (out and os allow it)
                if constexpr (F32OUT) {
                    *reinterpret_cast<f32x4 *>(static_cast<float *>(out) + i) = f32x4{v[0], v[1], v[2], v[3]};
                } else {
                    typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2;
                    *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(out) + i) =
                        u32x2{uint32_t(f2bf(v[0])) | uint32_t(f2bf(v[1])) << 16,
                              uint32_t(f2bf(v[2])) | uint32_t(f2bf(v[3])) << 16};
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (co + e >= cout) break;
                    if constexpr (F32OUT) static_cast<float *>(out)[i + e] = v[e];
                    else static_cast<uint16_t *>(out)[i + e] = f2bf(v[e]);
                }
            }
        }
    }
}

// 33 to 32 NC input channels, NC 2 to 4: the same tile with every channel of the
// block's pixels in LDS at once (rows of 64 NC + 16 bytes: as conflict-free), one
// block a CU, so that the sum still runs over the taps first and the channels
// within a tap (an activation rounds to the same bf16).  Measured in that step,
// operands from L1 before: 64 channels 155 -> 70 us on average, 96 -> 32 at the
// finest level 266 -> 181 us, 128 channels 50 us.
template <int KS, int NT, int NC, bool F32OUT>
__global__ void __launch_bounds__(256)
conv_lds_kernel(const uint16_t *__restrict__ in, int H, int W, int cin, int is, const uint16_t *__restrict__ w, int cout,
                const float *__restrict__ bias, int relu, void *__restrict__ out, int os, int ncot, int vec)
{
    constexpr int R = KS / 2, IW = 64 + 2 * R, IH = 4 + 2 * R, CO = 16 * NT, PT = 32 * NC + 8;
    constexpr int NI = IH * IW * 4 * NC, NW = KS * CO * 4 * NC;   // 16-byte units staged
    constexpr int UW = (NW + 255) / 256;
    __shared__ __attribute__((aligned(16))) uint16_t sI[IH * IW * PT];
    __shared__ __attribute__((aligned(16))) uint16_t sW[KS * CO * PT];
    const int tid = int(threadIdx.x), lane = tid & 63, wv = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int x0 = int(blockIdx.x) * 64, y0 = int(blockIdx.y) * 4;
    const int n = int(blockIdx.z) / ncot, co0 = (int(blockIdx.z) % ncot) * CO;
    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 rw[UW];
    auto fetch_w = [&](int dy) {   // the KS taps of row dy
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            const int k = tid + 256 * u, row = k / (4 * NC), ci = k % (4 * NC) * 8;
            const int dx = row / CO, co = co0 + row % CO;
            rw[u] = u32x4{0u, 0u, 0u, 0u};
            if (row < KS * CO && ci < cin && co < cout)
                rw[u] = *reinterpret_cast<const u32x4 *>(w + (int64_t(co) * (KS * KS) + dy * KS + dx) * cin + ci);
        }
    };
    fetch_w(0);
    // the pixels and their halo (zeros outside), eight loads in flight a thread
    // (unrolled whole, the loop was slower: 81, 234 and 55 us for 70, 181 and 50)
    for (int k0 = tid; k0 < NI; k0 += 256 * 8) {
        u32x4 ri[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = k0 + 256 * u, px = k / (4 * NC), ci = k % (4 * NC) * 8;
            const int y = y0 - R + px / IW, x = x0 - R + px % IW;
            ri[u] = u32x4{0u, 0u, 0u, 0u};
            if (k < NI && ci < cin && y >= 0 && y < H && x >= 0 && x < W)
                ri[u] = *reinterpret_cast<const u32x4 *>(in + ((int64_t(n) * H + y) * W + x) * is + ci);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = k0 + 256 * u;
            if (k < NI) *reinterpret_cast<u32x4 *>(sI + k / (4 * NC) * PT + k % (4 * NC) * 8) = ri[u];
        }
    }
#pragma unroll
    for (int dy = 0; dy < KS; ++dy) {
        if (dy > 0) __syncthreads();
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            const int k = tid + 256 * u;
            if (k < NW) *reinterpret_cast<u32x4 *>(sW + k / (4 * NC) * PT + k % (4 * NC) * 8) = rw[u];
        }
        __syncthreads();
        if (dy + 1 < KS) fetch_w(dy + 1);
#pragma unroll
        for (int dx = 0; dx < KS; ++dx)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                bf16x8 wf[NT], px[4];
#pragma unroll
                for (int t = 0; t < NT; ++t) wf[t] = ld8(sW + (dx * CO + 16 * t + r16) * PT + 32 * c + 8 * g);
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    px[m] = ld8(sI + ((wv + dy) * IW + 16 * m + r16 + dx) * PT + 32 * c + 8 * g);
#pragma unroll
                for (int m = 0; m < 4; ++m)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[m][t] = mma(wf[t], px[m], acc[m][t]);
            }
    }
    const int y = y0 + wv;
    if (y >= H) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + 16 * t + 4 * g;
        if (co >= cout) continue;
        float bv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[e] = bias && co + e < cout ? bias[co + e] : 0.f;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int x = x0 + 16 * m + r16;
            if (x >= W) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = acc[m][t][e] + bv[e];
                if (relu) v[e] = fmaxf(v[e], 0.f);
            }
            const int64_t i = ((int64_t(n) * H + y) * W + x) * os + co;
            if (vec && co + 4 <= cout) {   // four channels in one store (out and os allow it)
                if constexpr (F32OUT) {
                    *reinterpret_cast<f32x4 *>(static_cast<float *>(out) + i) = f32x4{v[0], v[1], v[2], v[3]};
                } else {
                    typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2;
                    *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(out) + i) =
                        u32x2{uint32_t(f2bf(v[0])) | uint32_t(f2bf(v[1])) << 16,
                              uint32_t(f2bf(v[2])) | uint32_t(f2bf(v[3])) << 16};
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (co + e >= cout) break;
                    if constexpr (F32OUT) static_cast<float *>(out)[i + e] = v[e];
                    else static_cast<uint16_t *>(out)[i + e] = f2bf(v[e]);
                }
            }
        }
    }
}

// More than 128 input channels.  Block: 4 waves, 128 consecutive pixels of one
// image row (32 per wave, two 16-row A tiles) x 16 NT output channels.
// Grid: (ceil(W / 128), H, N * ceil(cout / (16 NT))).  Every operand comes from
// L1 or L2; staging a chunk of the input for all taps instead would sum the
// chunks before the taps, and the network's bf16 activations then round apart.
template <int KS, int NT, bool F32OUT>
__global__ void __launch_bounds__(256) conv_fwd_kernel(const uint16_t *__restrict__ in, int H, int W, int cin,
                                                       int is, const uint16_t *__restrict__ w, int cout,
                                                       const float *__restrict__ bias, int relu,
                                                       void *__restrict__ out, int os, int ncot)
{
    const int lane = int(threadIdx.x) & 63, wv = int(threadIdx.x) >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int y = int(blockIdx.y);
    const int n = int(blockIdx.z) / ncot, co0 = (int(blockIdx.z) % ncot) * 16 * NT;
    const int x0 = int(blockIdx.x) * 128 + wv * 32;
    constexpr int R = KS / 2;
    const int nchunk = (cin + 31) / 32;
    f32x4 acc[2][NT];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int tap = 0; tap < KS * KS; ++tap) {
        const int sy = y + tap / KS - R, dx = tap % KS - R;
        const bool rowok = sy >= 0 && sy < H;
        const int64_t rowbase = (int64_t(n) * H + sy) * W;
        for (int c = 0; c < nchunk; ++c) {
            const int ci = c * 32 + 8 * g;
            const bool ciok = ci < cin;
            bf16x8 a[2], b[NT];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int sx = x0 + 16 * m + r16 + dx;
                a[m] = (rowok && ciok && sx >= 0 && sx < W) ? ld8(in + (rowbase + sx) * is + ci) : zero8();
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int co = co0 + 16 * t + r16;
                b[t] = (ciok && co < cout) ? ld8(w + (int64_t(co) * (KS * KS) + tap) * cin + ci) : zero8();
            }
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[m][t] = mma(a[m], b[t], acc[m][t]);
        }
    }
    const int64_t obase = (int64_t(n) * H + y) * W;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + 16 * t + r16;
        if (co >= cout) continue;
        const float bv = bias ? bias[co] : 0.f;
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int x = x0 + 16 * m + 4 * g + e;
                if (x >= W) continue;
                float v = acc[m][t][e] + bv;
                if (relu) v = fmaxf(v, 0.f);
                const int64_t i = (obase + x) * os + co;
                if constexpr (F32OUT) static_cast<float *>(out)[i] = v;
                else static_cast<uint16_t *>(out)[i] = f2bf(v);
            }
    }
}

// ---------------------------------------------------------------- weight gradient
// Block: 4 waves, 32 TO output x 32 TI input channels, every tap, over strips
// of SP columns and a segment of rows of an image: one strip, or several in turn
// where there are more of them than workgroups (wgrad_plan).  The contraction runs over
// pixels: each image row of the strip (input with its ks / 2 halo columns, dout
// without) is staged once in LDS as [pixel][channel] and feeds all ks * ks taps
// (the input rows of a window stay in a ring), where ds_read_b64_tr_b16 hands a
// lane four pixels of its channel: a 16-lane group reads 4 pixels x 16 channels
// and gets them transposed.  The same pixel order in both operands is all the
// product needs, so lane group g takes pixels 4g.. and 16 + 4g.. of a 32-pixel
// step, and a tap's shift is a pixel offset.  A wave owns a 32 x 32 channel tile
// of all taps (144 accumulators at 3 x 3); a block of fewer than four channel
// tiles gives the other waves (WK) pixels of their own.  Row pitches of 80 and 48
// halves put 8 consecutive pixels' 32 bytes on different banks.  The next rows'
// loads are in flight while a row is multiplied, one barrier a row.
//
// Measured in a 2 x 384 x 1152, 4-level, base-32 training step (14 layers, 285
// GFLOP): 22 to 83 us a layer, 33.5 us on average at 64 x 64 tiles; one block a
// tap, each staging both operands again through 2-byte transposing LDS stores,
// took 395 us on average.  Bound by the LDS reads (80 transposing reads a wave
// and row against 72 MFMAs).
template <int KS, int TO, int TI>
struct WgradTile {
    static constexpr int WK = 4 / (TO * TI);
    static constexpr int KPW = WK == 1 ? 64 : 32;    // pixels a wave takes of a row
    static constexpr int SP = KPW * WK;              // strip columns
    static constexpr int R = KS / 2;
    static constexpr int NS = KS == 3 ? 4 : 2;       // input rows kept
    static constexpr int PI = TI == 2 ? 80 : 48, PD = TO == 2 ? 80 : 48;
    static constexpr int IW = SP + 2 * R;
    static constexpr int UI = (IW * TI * 4 + 255) / 256, UD = (SP * TO * 4 + 255) / 256;   // 16-byte units a thread
};

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;

__device__ __forceinline__ bf16x8 ld_tr(const uint16_t *p, int pitch)
{
    struct Pair {
        s16x4 lo, hi;
    } v;
    using L = __attribute__((address_space(3))) s16x4;
    v.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)(p));
    v.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)(p + 16 * pitch));
    return __builtin_bit_cast(bf16x8, v);
}

template <int KS, int TO, int TI>
__global__ void __launch_bounds__(256, 2) wgrad_kernel(const uint16_t *__restrict__ in, int H, int W, int cin, int is,
                                                       const uint16_t *__restrict__ dout, int cout, int ds,
                                                       float *__restrict__ partials, int nsx, int nsy, int rows,
                                                       int strips)
{
    using T = WgradTile<KS, TO, TI>;
    __shared__ __attribute__((aligned(16))) uint16_t mem[T::NS * T::IW * T::PI + 2 * T::SP * T::PD];
    auto sI = [&](int y) { return mem + (y + T::NS) % T::NS * (T::IW * T::PI); };
    auto sD = [&](int y) { return mem + T::NS * T::IW * T::PI + (y & 1) * (T::SP * T::PD); };
    const int tid = int(threadIdx.x), lane = tid & 63, wv = tid >> 6;
    const int g = lane >> 4, i16 = lane & 15;
    const int ci0 = int(blockIdx.y) * 32 * TI, co0 = int(blockIdx.z) * 32 * TO;
    const int wk = wv / (TO * TI), wo = wv % (TO * TI) / TI, wi = wv % TI;

    f32x4 acc[KS * KS][2][2];
#pragma unroll
    for (int t = 0; t < KS * KS; ++t)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[t][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    int n = 0, x0 = 0, ye = 0;   // the strip's image, first column and row end
    u32x4 ri[T::UI], rd[T::UD];
    auto fetch_in = [&](int y) {   // input row y (zeros outside the image)
#pragma unroll
        for (int u = 0; u < T::UI; ++u) {
            const int k = tid + 256 * u, px = k / (TI * 4), c = ci0 + k % (TI * 4) * 8, x = x0 - T::R + px;
            ri[u] = u32x4{0u, 0u, 0u, 0u};
            if (px < T::IW && c < cin && y >= 0 && y < H && x >= 0 && x < W)
                ri[u] = *reinterpret_cast<const u32x4 *>(in + ((int64_t(n) * H + y) * W + x) * is + c);
        }
    };
    auto fetch_dout = [&](int y) {
#pragma unroll
        for (int u = 0; u < T::UD; ++u) {
            const int k = tid + 256 * u, px = k / (TO * 4), c = co0 + k % (TO * 4) * 8, x = x0 + px;
            rd[u] = u32x4{0u, 0u, 0u, 0u};
            if (px < T::SP && c < cout && y < ye && x < W)
                rd[u] = *reinterpret_cast<const u32x4 *>(dout + ((int64_t(n) * H + y) * W + x) * ds + c);
        }
    };
    auto put_in = [&](int y) {
        uint16_t *d = sI(y);
#pragma unroll
        for (int u = 0; u < T::UI; ++u) {
            const int k = tid + 256 * u, px = k / (TI * 4);
            if (px < T::IW) *reinterpret_cast<u32x4 *>(d + px * T::PI + k % (TI * 4) * 8) = ri[u];
        }
    };
    auto put_dout = [&](int y) {
        uint16_t *d = sD(y);
#pragma unroll
        for (int u = 0; u < T::UD; ++u) {
            const int k = tid + 256 * u, px = k / (TO * 4);
            if (px < T::SP) *reinterpret_cast<u32x4 *>(d + px * T::PD + k % (TO * 4) * 8) = rd[u];
        }
    };
    const int fp = 4 * g + i16 / 4, fc = 4 * (i16 % 4);   // a lane's pixel and channel within a fragment
    for (int u = int(blockIdx.x); u < strips; u += int(gridDim.x)) {
        const int yb = u / nsx % nsy * rows;
        n = u / (nsx * nsy);
        x0 = u % nsx * T::SP;
        ye = std::min(yb + rows, H);
        if (u != int(blockIdx.x)) __syncthreads();   // the rows of the strip before are still read
        for (int y = yb - T::R; y <= yb + T::R; ++y) {
            fetch_in(y);
            put_in(y);
        }
        fetch_dout(yb);
        put_dout(yb);
        for (int y = yb; y < ye; ++y) {
            __syncthreads();
            fetch_in(y + T::R + 1);
            fetch_dout(y + 1);
#pragma unroll
            for (int k = 0; k < T::KPW / 32; ++k) {
                const int p = wk * T::KPW + 32 * k + fp;
                bf16x8 A[2];
#pragma unroll
                for (int a = 0; a < 2; ++a) A[a] = ld_tr(sD(y) + p * T::PD + wo * 32 + 16 * a + fc, T::PD);
#pragma unroll
                for (int dy = 0; dy < KS; ++dy) {
                    const uint16_t *row = sI(y + dy - T::R) + wi * 32 + fc;
#pragma unroll
                    for (int dx = 0; dx < KS; ++dx) {
#pragma unroll
                        for (int b = 0; b < 2; ++b) {
                            const bf16x8 Bv = ld_tr(row + (p + dx) * T::PI + 16 * b, T::PI);
#pragma unroll
                            for (int a = 0; a < 2; ++a) acc[dy * KS + dx][a][b] = mma(A[a], Bv, acc[dy * KS + dx][a][b]);
                        }
                    }
                }
            }
            put_in(y + T::R + 1);
            put_dout(y + 1);
        }
    }
    // the waves of one channel tile (WK of them) meet in LDS, a tap at a time;
    // each then writes 4 / WK of the tile's four 16 x 16 parts
    f32x4 *red = reinterpret_cast<f32x4 *>(mem);
#pragma unroll
    for (int t = 0; t < KS * KS; ++t) {
        float *dst = partials + (int64_t(blockIdx.x) * (KS * KS) + t) * cout * cin;
        if constexpr (T::WK > 1) {
            __syncthreads();
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) red[(wv * 4 + 2 * a + b) * 64 + lane] = acc[t][a][b];
            __syncthreads();
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                f32x4 v = acc[t][a][b];
                if constexpr (T::WK > 1) {
                    if ((2 * a + b) % T::WK != wk) continue;
                    v = red[((wv - wk * (TO * TI)) * 4 + 2 * a + b) * 64 + lane];
#pragma unroll
                    for (int k = 1; k < T::WK; ++k) v += red[((wv + (k - wk) * (TO * TI)) * 4 + 2 * a + b) * 64 + lane];
                }
                const int ci = ci0 + wi * 32 + 16 * b + i16;
                if (ci >= cin) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int co = co0 + wo * 32 + 16 * a + 4 * g + e;
                    if (co < cout) dst[int64_t(co) * cin + ci] = v[e];
                }
            }
    }
}

// dw[co, tap, ci] = sum over splits of partials[split, tap, co, ci].  A block
// takes 32 consecutive values of the partials' order; its 8 groups of 32 lanes
// stride the splits and meet in LDS, always in the same order.  (One thread a
// value, walking up to 4096 splits alone, took 423 us a layer.)
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float *__restrict__ partials, int splits, int taps,
                                                           int cout, int cin, float *__restrict__ dw)
{
    __shared__ float red[256];
    const int64_t n = int64_t(taps) * cout * cin;
    const int64_t k = int64_t(blockIdx.x) * 32 + (threadIdx.x & 31);
    float s = 0.f;
    if (k < n) {
#pragma unroll 4
        for (int sp = int(threadIdx.x) >> 5; sp < splits; sp += 8) s += partials[int64_t(sp) * n + k];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x >= 32 || k >= n) return;
    for (int j = 1; j < 8; ++j) s += red[threadIdx.x + 32 * j];
    const int ci = int(k % cin);
    const int64_t t2 = k / cin;
    const int co = int(t2 % cout), tap = int(t2 / cout);
    dw[(int64_t(co) * taps + tap) * cin + ci] = s;
}

// partial[split, c] = sum over the split's pixels of x[p, c]; then out[c].
// Thread t takes channel c0 + t % CB and pixel sub-lane t / CB (J = 256 / CB
// sub-lanes stride the split's pixels), the J lane sums meet in LDS.
__global__ void __launch_bounds__(256) colsum_kernel(const uint16_t *__restrict__ x, int xs, int C, int64_t P,
                                                     int64_t per, float *__restrict__ partial)
{
    __shared__ float red[256];
    const int64_t pb = int64_t(blockIdx.x) * per, pe = std::min(P, pb + per);
    const int CB = C < 256 ? C : 256;
    const int J = 256 / CB;
    const int t = int(threadIdx.x), j = t / CB, cl = t % CB;
    for (int c0 = 0; c0 < C; c0 += CB) {
        const int c = c0 + cl;
        float s = 0.f;
        if (j < J && c < C)
            for (int64_t p = pb + j; p < pe; p += J) s += bf2f(x[p * xs + c]);
        red[t] = s;
        __syncthreads();
        if (j == 0 && c < C) {
            float tot = 0.f;
            for (int k = 0; k < J; ++k) tot += red[k * CB + cl];
            partial[int64_t(blockIdx.x) * C + c] = tot;
        }
        __syncthreads();
    }
}

// One block per channel: a fixed-order tree over the splits.
__global__ void __launch_bounds__(256) colsum_reduce_kernel(const float *__restrict__ partial, int splits, int C,
                                                            float *__restrict__ out)
{
    __shared__ float red[256];
    const int c = int(blockIdx.x);
    float s = 0.f;
    for (int sp = int(threadIdx.x); sp < splits; sp += 256) s += partial[int64_t(sp) * C + c];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (int(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[c] = red[0];
}

__global__ void __launch_bounds__(256) flip_kernel(const uint16_t *__restrict__ w, int cout, int cin, int taps,
                                                   uint16_t *__restrict__ wt)
{
    const int64_t n = int64_t(cout) * taps * cin;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        // i indexes wt[ci, tap, co]
        const int co = int(i % cout);
        const int64_t t2 = i / cout;
        const int tap = int(t2 % taps), ci = int(t2 / taps);
        wt[i] = w[(int64_t(co) * taps + (taps - 1 - tap)) * cin + ci];
    }
}

// ---------------------------------------------------------------- element-wise
__global__ void __launch_bounds__(256) relu_bwd_kernel(uint16_t *__restrict__ d, int dsd,
                                                       const uint16_t *__restrict__ act, int as, int64_t P, int C)
{
    const int64_t n = P * C;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const int64_t p = i / C;
        const int c = int(i % C);
        if (!(bf2f(act[p * as + c]) > 0.f)) d[p * dsd + c] = 0;
    }
}

// H, W: the input (fine) extents.
__global__ void __launch_bounds__(256) pool2_fwd_kernel(const uint16_t *__restrict__ in, int is, int N, int H, int W,
                                                        int C, uint16_t *__restrict__ out, int os)
{
    const int Ho = H / 2, Wo = W / 2;
    const int64_t n = int64_t(N) * Ho * Wo * C;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const int c = int(i % C);
        const int64_t q = i / C;
        const int xo = int(q % Wo), yo = int((q / Wo) % Ho);
        const int64_t nn = q / (int64_t(Wo) * Ho);
        const int64_t p00 = (nn * H + 2 * yo) * W + 2 * xo;
        const float s = (bf2f(in[p00 * is + c]) + bf2f(in[(p00 + 1) * is + c])) +
                        (bf2f(in[(p00 + W) * is + c]) + bf2f(in[(p00 + W + 1) * is + c]));
        out[q * os + c] = f2bf(0.25f * s);
    }
}

__global__ void __launch_bounds__(256) pool2_bwd_kernel(const uint16_t *__restrict__ dout, int dsd, int N, int H,
                                                        int W, int C, uint16_t *__restrict__ din, int dis)
{
    const int Ho = H / 2, Wo = W / 2;
    const int64_t n = int64_t(N) * H * W * C;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const int c = int(i % C);
        const int64_t p = i / C;
        const int x = int(p % W), y = int((p / W) % H);
        const int64_t nn = p / (int64_t(W) * H);
        const int64_t q = (nn * Ho + y / 2) * Wo + x / 2;
        din[p * dis + c] = f2bf(bf2f(din[p * dis + c]) + 0.25f * bf2f(dout[q * dsd + c]));
    }
}

// H, W: the coarse (input) extents.
__global__ void __launch_bounds__(256) up2_fwd_kernel(const uint16_t *__restrict__ in, int is, int N, int H, int W,
                                                      int C, uint16_t *__restrict__ out, int os)
{
    const int Hf = 2 * H, Wf = 2 * W;
    const int64_t n = int64_t(N) * Hf * Wf * C;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const int c = int(i % C);
        const int64_t p = i / C;
        const int x = int(p % Wf), y = int((p / Wf) % Hf);
        const int64_t nn = p / (int64_t(Wf) * Hf);
        out[p * os + c] = in[((nn * H + y / 2) * W + x / 2) * is + c];
    }
}

__global__ void __launch_bounds__(256) up2_bwd_kernel(const uint16_t *__restrict__ dout, int dsd, int N, int H, int W,
                                                      int C, uint16_t *__restrict__ din, int dis)
{
    const int Wf = 2 * W;
    const int64_t n = int64_t(N) * H * W * C;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const int c = int(i % C);
        const int64_t q = i / C;
        const int x = int(q % W), y = int((q / W) % H);
        const int64_t nn = q / (int64_t(W) * H);
        const int64_t f00 = (nn * 2 * H + 2 * y) * Wf + 2 * x;
        const float s = (bf2f(dout[f00 * dsd + c]) + bf2f(dout[(f00 + 1) * dsd + c])) +
                        (bf2f(dout[(f00 + Wf) * dsd + c]) + bf2f(dout[(f00 + Wf + 1) * dsd + c]));
        din[q * dis + c] = f2bf(s);
    }
}

// The same passes on eight channels (16 bytes) a thread, for views whose
// channels and strides are multiples of 8 on 16-byte aligned pointers, with a
// 32-bit index.  One channel a thread spent its time on 64-bit divisions and
// 2-byte accesses: in a 2 x 384 x 1152, base-32 training step relu 25, upsample
// 106 / 39, pool 22 / 62, column sum 34 us a call.
__device__ __forceinline__ void unpack8(const u32x4 v, float (&f)[8])
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        f[2 * e] = bf2f(uint16_t(v[e] & 0xffffu));
        f[2 * e + 1] = bf2f(uint16_t(v[e] >> 16));
    }
}
__device__ __forceinline__ u32x4 pack8(const float (&f)[8])
{
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = uint32_t(f2bf(f[2 * e])) | uint32_t(f2bf(f[2 * e + 1])) << 16;
    return v;
}
__device__ __forceinline__ u32x4 at8(const uint16_t *p, int64_t i) { return *reinterpret_cast<const u32x4 *>(p + i); }
__device__ __forceinline__ void put8(uint16_t *p, int64_t i, u32x4 v) { *reinterpret_cast<u32x4 *>(p + i) = v; }

__global__ void __launch_bounds__(256) relu_bwd8_kernel(uint16_t *__restrict__ d, int dsd,
                                                        const uint16_t *__restrict__ act, int as, unsigned n, unsigned C8)
{
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const int64_t p = i / C8;
        const int c = int(i % C8) * 8;
        float a[8];
        unpack8(at8(act, p * as + c), a);
        u32x4 v = at8(d, p * dsd + c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            v[e] &= (a[2 * e] > 0.f ? 0xffffu : 0u) | (a[2 * e + 1] > 0.f ? 0xffff0000u : 0u);
        put8(d, p * dsd + c, v);
    }
}

// Coarse pixel q of (H, W) per (image): the fine pixel at its corner.
__device__ __forceinline__ int64_t fine00(unsigned q, int H, int W)
{
    const unsigned x = q % unsigned(W), r = q / unsigned(W), y = r % unsigned(H), nn = r / unsigned(H);
    return (int64_t(nn) * 2 * H + 2 * y) * (2 * int64_t(W)) + 2 * x;
}

// MODE 0: upsample (coarse -> fine); 1: its adjoint; 2: average pool (fine ->
// coarse); 3: its adjoint, added into the fine gradient.  H, W: coarse extents.
template <int MODE>
__global__ void __launch_bounds__(256) scale2_kernel(uint16_t *__restrict__ coarse, int cs, uint16_t *__restrict__ fine,
                                                     int fs, int H, int W, unsigned n, unsigned C8)
{
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const unsigned q = i / C8;
        const int c = int(i % C8) * 8;
        const int64_t f00 = fine00(q, H, W), W2 = 2 * int64_t(W);
        const int64_t at[4] = {f00 * fs + c, (f00 + 1) * fs + c, (f00 + W2) * fs + c, (f00 + W2 + 1) * fs + c};
        const int64_t ac = int64_t(q) * cs + c;
        if constexpr (MODE == 0) {
            const u32x4 v = at8(coarse, ac);
#pragma unroll
            for (int k = 0; k < 4; ++k) put8(fine, at[k], v);
        } else if constexpr (MODE == 3) {
            float d[8];
            unpack8(at8(coarse, ac), d);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float f[8];
                unpack8(at8(fine, at[k]), f);
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = f[e] + 0.25f * d[e];
                put8(fine, at[k], pack8(f));
            }
        } else {
            float f[4][8], o[8];
#pragma unroll
            for (int k = 0; k < 4; ++k) unpack8(at8(fine, at[k]), f[k]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float sum = (f[0][e] + f[1][e]) + (f[2][e] + f[3][e]);
                o[e] = MODE == 2 ? 0.25f * sum : sum;
            }
            put8(coarse, ac, pack8(o));
        }
    }
}

// Column sums on eight channels a thread (C a multiple of 8, at most 2048).
__global__ void __launch_bounds__(256) colsum8_kernel(const uint16_t *__restrict__ x, int xs, int C, int64_t P,
                                                      int64_t per, float *__restrict__ partial)
{
    __shared__ float red[256][9];
    const int64_t pb = int64_t(blockIdx.x) * per, pe = std::min(P, pb + per);
    const int C8 = C / 8, J = 256 / C8, t = int(threadIdx.x), j = t / C8, cl = t % C8;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (j < J)
        for (int64_t p = pb + j; p < pe; p += J) {
            float f[8];
            unpack8(at8(x, p * xs + cl * 8), f);
#pragma unroll
            for (int e = 0; e < 8; ++e) s[e] += f[e];
        }
#pragma unroll
    for (int e = 0; e < 8; ++e) red[t][e] = s[e];
    __syncthreads();
    for (int c = t; c < C; c += 256) {
        float tot = 0.f;
        for (int k = 0; k < J; ++k) tot += red[k * C8 + c / 8][c % 8];
        partial[int64_t(blockIdx.x) * C + c] = tot;
    }
}

struct Planes {
    const float *p[4];
    float s[4];
};

__global__ void __launch_bounds__(256) pack_input_kernel(Planes pl, int nsrc, int64_t P, uint16_t *__restrict__ x,
                                                         int xs)
{
    const int64_t n = P * xs;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const int c = int(i % xs);
        const int64_t p = i / xs;
        float v = 0.f;
        if (c < nsrc) v = pl.s[c] * pl.p[c][p];
        x[i] = f2bf(v);
    }
}

__global__ void __launch_bounds__(256) mse_kernel(const float *__restrict__ out, int os, const float *__restrict__ tgt,
                                                  const float *__restrict__ mask, int64_t P, double count,
                                                  uint16_t *__restrict__ dout, int dsd, double *__restrict__ partial)
{
    __shared__ double red[256];
    double acc = 0.0;
    const float sc = float(2.0 / count);
    for (int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x; p < P; p += int64_t(gridDim.x) * 256) {
        const float r = out[p * os] - tgt[p];
        const float m = mask ? mask[p] : 1.f;
        acc += double(r) * double(r) * double(m);
        dout[p * dsd] = f2bf(sc * r * m);
        for (int c = 1; c < dsd; ++c) dout[p * dsd + c] = 0;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (int(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) sum_kernel(const double *__restrict__ partial, int np, double scale,
                                                  double *__restrict__ out)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (int i = int(threadIdx.x); i < np; i += 256) acc += partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (int(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = scale * red[0];
}

__global__ void __launch_bounds__(256) adam_kernel(float *__restrict__ w, const float *__restrict__ g,
                                                   float *__restrict__ m, float *__restrict__ v,
                                                   uint16_t *__restrict__ wbf, int64_t n, float lr, float b1,
                                                   float b2, float eps, float c1, float c2)
{
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = wi;
        if (wbf) wbf[i] = f2bf(wi);
    }
}

__global__ void __launch_bounds__(256) to_bf16_kernel(const float *__restrict__ s, uint16_t *__restrict__ d, int64_t n)
{
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) d[i] = f2bf(s[i]);
}

unsigned blocks_for(int64_t n) { return unsigned(std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 16384))); }

// Whether a pass over n8 groups of 8 channels can run 16 bytes a thread.  The
// kernels count in 32 bits unsigned; a negative extent stays with the 64-bit
// passes, which do nothing for it.
bool vec8(int C, int64_t n8, const void *a, int as, const void *b, int bs)
{
    return C % 8 == 0 && as % 8 == 0 && bs % 8 == 0 &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0 && n8 >= 0 && n8 < (int64_t(1) << 31);
}

void check_view(const void *p, int stride, int channels, const char *what)
{
    SWP_CHECK(p != nullptr, what, ": null pointer");
    SWP_CHECK((reinterpret_cast<uintptr_t>(p) & 15) == 0, what, ": pointer not 16-byte aligned");
    SWP_CHECK(stride % 8 == 0 && channels % 8 == 0 && channels <= stride && channels > 0, what,
              ": channels (", channels, ") and stride (", stride, ") must be positive multiples of 8, channels <= stride");
}

// The weight gradient's launch: 64 channels a tile where the count is a multiple
// of 64, else 32; rows a segment so that at most kWgradBlocks workgroups run (two
// fit on each of the 256 CUs) where that leaves at least 4.  Where whole columns
// of many images are still more strips than that, a workgroup takes several, cut
// so that all have about as many rows: every workgroup writes a partial tile of
// all taps, which the reduce pass reads again, so the scratch holds at most
// kWgradBlocks of them (75 MB at 64 x 64 channels and 3 x 3) or, past 512 channel
// tiles, one for each.  Measured with one strip a workgroup / as now: 16 x 48 x
// 144, 256 channels both ways 179 / 166 us (114 / 76 MB), 64 images 735 / 593 (454 / 76),
// 16 x 24 x 72, 512 channels 276 / 217 (303 / 77).
constexpr int64_t kWgradBlocks = 512;

struct WgradPlan {
    int to, ti, nsx, nsy, rows, strips, blocks;
};

WgradPlan wgrad_plan(int N, int H, int W, int cin, int cout)
{
    WgradPlan p{};
    p.to = cout % 64 == 0 ? 2 : 1;
    p.ti = cin % 64 == 0 ? 2 : 1;
    const int wk = 4 / (p.to * p.ti), sp = wk == 4 ? 128 : 64;
    const int64_t tiles = int64_t((cin + 32 * p.ti - 1) / (32 * p.ti)) * ((cout + 32 * p.to - 1) / (32 * p.to));
    p.nsx = (W + sp - 1) / sp;
    const int64_t most = std::max<int64_t>(1, kWgradBlocks / tiles);   // workgroups a channel tile
    const int64_t cols = int64_t(p.nsx) * N;
    if (cols <= most) {
        const int64_t want = std::max<int64_t>(1, kWgradBlocks / (tiles * cols));
        p.rows = int(std::max<int64_t>(std::min(H, 4), (H + want - 1) / want));
    } else {
        int64_t best = INT64_MAX;   // rows that the busiest workgroup walks, two more each strip
        for (int k = 1; k <= 8 && (k == 1 || H / k >= 4); ++k) {
            const int rows = (H + k - 1) / k;
            const int64_t cost = (cols * ((H + rows - 1) / rows) + most - 1) / most * (rows + 2);
            if (cost < best) {
                best = cost;
                p.rows = rows;
            }
        }
    }
    p.nsy = (H + p.rows - 1) / p.rows;
    p.strips = p.nsx * p.nsy * N;
    const int64_t each = (p.strips + most - 1) / most;
    p.blocks = int((p.strips + each - 1) / each);
    return p;
}

constexpr int kColSplits = 512;

}  // namespace

void conv_fwd(const uint16_t *in, int N, int H, int W, int cin, int in_stride, const uint16_t *w, int cout, int ks,
              const float *bias, bool relu, void *out, int out_stride, bool out_f32)
{
    SWP_CHECK(ks == 1 || ks == 3, "conv: kernel size must be 1 or 3");
    SWP_CHECK(N >= 1 && H >= 1 && W >= 1 && N * int64_t((cout + 63) / 64) <= 65535 && H <= 65535,
              "conv: bad extents");
    check_view(in, in_stride, cin, "conv input");
    SWP_CHECK(w && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "conv: weights null or not 16-byte aligned");
    SWP_CHECK(out && cout >= 1 && cout <= out_stride, "conv: bad output view");
    const int nt = cout > 32 ? 4 : cout > 16 ? 2 : 1;
    const int ncot = (cout + 16 * nt - 1) / (16 * nt);
    const int r = relu ? 1 : 0;
    const int vec = out_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & (out_f32 ? 15 : 7)) == 0;
    const dim3 grid(unsigned((W + 127) / 128), unsigned(H), unsigned(N * ncot));
    const dim3 grid_lds(unsigned((W + 63) / 64), unsigned((H + 3) / 4), unsigned(N * ncot));
#define SWP_CONV_LDS(KS, NT, NC, F32)                                                                             \
    hipLaunchKernelGGL((conv_lds_kernel<KS, NT, NC, F32>), grid_lds, dim3(256), 0, stream(), in, H, W, cin,       \
                       in_stride, w, cout, bias, r, out, out_stride, ncot, vec)
#define SWP_CONV_LAUNCH(KS, NT, F32)                                                                              \
    do {                                                                                                          \
        if (cin <= 32)                                                                                            \
            hipLaunchKernelGGL((conv_c32_kernel<KS, NT, F32>), grid_lds, dim3(256), 0, stream(), in, H, W, cin,   \
                               in_stride, w, cout, bias, r, out, out_stride, ncot, vec);                          \
        else if (cin <= 64) SWP_CONV_LDS(KS, NT, 2, F32);                                                         \
        else if (cin <= 96) SWP_CONV_LDS(KS, NT, 3, F32);                                                         \
        else if (cin <= 128) SWP_CONV_LDS(KS, NT, 4, F32);                                                        \
        else                                                                                                      \
            hipLaunchKernelGGL((conv_fwd_kernel<KS, NT, F32>), grid, dim3(256), 0, stream(), in, H, W, cin,       \
                               in_stride, w, cout, bias, r, out, out_stride, ncot);                               \
    } while (0)
#define SWP_CONV_NT(KS, F32)                         \
    do {                                             \
        if (nt == 4) SWP_CONV_LAUNCH(KS, 4, F32);    \
        else if (nt == 2) SWP_CONV_LAUNCH(KS, 2, F32); \
        else SWP_CONV_LAUNCH(KS, 1, F32);            \
    } while (0)
    if (ks == 3) {
        if (out_f32) SWP_CONV_NT(3, true);
        else SWP_CONV_NT(3, false);
    } else {
        if (out_f32) SWP_CONV_NT(1, true);
        else SWP_CONV_NT(1, false);
    }
#undef SWP_CONV_NT
#undef SWP_CONV_LDS
#undef SWP_CONV_LAUNCH
    SWP_LAUNCHED();
}

int64_t conv_wgrad_partials(int N, int H, int W, int cin, int cout, int ks)
{
    return int64_t(wgrad_plan(N, H, W, cin, cout).blocks) * ks * ks * cout * cin + int64_t(kColSplits) * cout;
}

void conv_wgrad(const uint16_t *in, int N, int H, int W, int cin, int in_stride, const uint16_t *dout, int cout,
                int dout_stride, int ks, float *dw, float *db, float *partials)
{
    SWP_CHECK(ks == 1 || ks == 3, "wgrad: kernel size must be 1 or 3");
    SWP_CHECK(N >= 1 && H >= 1 && W >= 1, "wgrad: bad extents");
    check_view(in, in_stride, cin, "wgrad input");
    check_view(dout, dout_stride, cout, "wgrad dout");
    SWP_CHECK(dw && partials, "wgrad: null output or scratch");
    const int64_t P = int64_t(N) * H * W;
    const WgradPlan w = wgrad_plan(N, H, W, cin, cout);
    const int splits = w.blocks;
    const dim3 grid(unsigned(w.blocks), unsigned((cin + 32 * w.ti - 1) / (32 * w.ti)),
                    unsigned((cout + 32 * w.to - 1) / (32 * w.to)));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream(), in, H, W, cin, in_stride, dout, cout, dout_stride,
                           partials, w.nsx, w.nsy, w.rows, w.strips);
    };
    const int tile = (w.to - 1) * 2 + w.ti - 1;
    if (ks == 3)
        tile == 3 ? launch(wgrad_kernel<3, 2, 2>) : tile == 2 ? launch(wgrad_kernel<3, 2, 1>)
            : tile == 1 ? launch(wgrad_kernel<3, 1, 2>) : launch(wgrad_kernel<3, 1, 1>);
    else
        tile == 3 ? launch(wgrad_kernel<1, 2, 2>) : tile == 2 ? launch(wgrad_kernel<1, 2, 1>)
            : tile == 1 ? launch(wgrad_kernel<1, 1, 2>) : launch(wgrad_kernel<1, 1, 1>);
    SWP_LAUNCHED();
    const int64_t n = int64_t(ks) * ks * cout * cin;
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(unsigned((n + 31) / 32)), dim3(256), 0, stream(), partials, splits, ks * ks,
                       cout, cin, dw);
    SWP_LAUNCHED();
    if (db) {
        float *cp = partials + int64_t(splits) * ks * ks * cout * cin;
        const int64_t cper = (P + kColSplits - 1) / kColSplits;
        if (cout <= 2048)
            hipLaunchKernelGGL(colsum8_kernel, dim3(kColSplits), dim3(256), 0, stream(), dout, dout_stride, cout, P, cper,
                               cp);
        else
            hipLaunchKernelGGL(colsum_kernel, dim3(kColSplits), dim3(256), 0, stream(), dout, dout_stride, cout, P, cper,
                               cp);
        SWP_LAUNCHED();
        hipLaunchKernelGGL(colsum_reduce_kernel, dim3(unsigned(cout)), dim3(256), 0, stream(), cp, kColSplits, cout,
                           db);
        SWP_LAUNCHED();
    }
}

void conv_flip(const uint16_t *w, int cout, int cin, int ks, uint16_t *wt)
{
    SWP_CHECK(w && wt && w != wt, "flip: bad buffers");
    const int64_t n = int64_t(cout) * ks * ks * cin;
    hipLaunchKernelGGL(flip_kernel, dim3(blocks_for(n)), dim3(256), 0, stream(), w, cout, cin, ks * ks, wt);
    SWP_LAUNCHED();
}

void relu_bwd(uint16_t *d, int d_stride, const uint16_t *act, int act_stride, int64_t P, int C)
{
    SWP_CHECK(d && act && C >= 1 && C <= d_stride && C <= act_stride, "relu_bwd: bad views");
    if (vec8(C, P * C / 8, d, d_stride, act, act_stride)) {
        hipLaunchKernelGGL(relu_bwd8_kernel, dim3(blocks_for(P * C / 8)), dim3(256), 0, stream(), d, d_stride, act,
                           act_stride, unsigned(P * C / 8), unsigned(C / 8));
        SWP_LAUNCHED();
        return;
    }
    hipLaunchKernelGGL(relu_bwd_kernel, dim3(blocks_for(P * C)), dim3(256), 0, stream(), d, d_stride, act,
                       act_stride, P, C);
    SWP_LAUNCHED();
}

void pool2_fwd(const uint16_t *in, int in_stride, int N, int H, int W, int C, uint16_t *out, int out_stride)
{
    SWP_CHECK(H % 2 == 0 && W % 2 == 0, "pool2: extents must be even");
    SWP_CHECK(in && out && C <= in_stride && C <= out_stride, "pool2: bad views");
    if (const int64_t n8 = int64_t(N) * (H / 2) * (W / 2) * (C / 8); vec8(C, n8, out, out_stride, in, in_stride)) {
        hipLaunchKernelGGL(scale2_kernel<2>, dim3(blocks_for(n8)), dim3(256), 0, stream(), const_cast<uint16_t *>(out),
                           out_stride, const_cast<uint16_t *>(in), in_stride, H / 2, W / 2, unsigned(n8), unsigned(C / 8));
        SWP_LAUNCHED();
        return;
    }
    hipLaunchKernelGGL(pool2_fwd_kernel, dim3(blocks_for(int64_t(N) * H * W * C / 4)), dim3(256), 0, stream(), in,
                       in_stride, N, H, W, C, out, out_stride);
    SWP_LAUNCHED();
}

void pool2_bwd_acc(const uint16_t *dout, int dout_stride, int N, int H, int W, int C, uint16_t *din, int din_stride)
{
    SWP_CHECK(H % 2 == 0 && W % 2 == 0, "pool2: extents must be even");
    SWP_CHECK(dout && din && C <= dout_stride && C <= din_stride, "pool2: bad views");
    if (const int64_t n8 = int64_t(N) * (H / 2) * (W / 2) * (C / 8); vec8(C, n8, dout, dout_stride, din, din_stride)) {
        hipLaunchKernelGGL(scale2_kernel<3>, dim3(blocks_for(n8)), dim3(256), 0, stream(), const_cast<uint16_t *>(dout),
                           dout_stride, const_cast<uint16_t *>(din), din_stride, H / 2, W / 2, unsigned(n8), unsigned(C / 8));
        SWP_LAUNCHED();
        return;
    }
    hipLaunchKernelGGL(pool2_bwd_kernel, dim3(blocks_for(int64_t(N) * H * W * C)), dim3(256), 0, stream(), dout,
                       dout_stride, N, H, W, C, din, din_stride);
    SWP_LAUNCHED();
}

void up2_fwd(const uint16_t *in, int in_stride, int N, int H, int W, int C, uint16_t *out, int out_stride)
{
    SWP_CHECK(in && out && C <= in_stride && C <= out_stride, "up2: bad views");
    if (const int64_t n8 = int64_t(N) * H * W * (C / 8); vec8(C, n8, in, in_stride, out, out_stride)) {
        hipLaunchKernelGGL(scale2_kernel<0>, dim3(blocks_for(n8)), dim3(256), 0, stream(), const_cast<uint16_t *>(in),
                           in_stride, const_cast<uint16_t *>(out), out_stride, H, W, unsigned(n8), unsigned(C / 8));
        SWP_LAUNCHED();
        return;
    }
    hipLaunchKernelGGL(up2_fwd_kernel, dim3(blocks_for(int64_t(N) * H * W * C * 4)), dim3(256), 0, stream(), in,
                       in_stride, N, H, W, C, out, out_stride);
    SWP_LAUNCHED();
}

void up2_bwd(const uint16_t *dout, int dout_stride, int N, int H, int W, int C, uint16_t *din, int din_stride)
{
    SWP_CHECK(dout && din && C <= dout_stride && C <= din_stride, "up2: bad views");
    if (const int64_t n8 = int64_t(N) * H * W * (C / 8); vec8(C, n8, din, din_stride, dout, dout_stride)) {
        hipLaunchKernelGGL(scale2_kernel<1>, dim3(blocks_for(n8)), dim3(256), 0, stream(), const_cast<uint16_t *>(din),
                           din_stride, const_cast<uint16_t *>(dout), dout_stride, H, W, unsigned(n8), unsigned(C / 8));
        SWP_LAUNCHED();
        return;
    }
    hipLaunchKernelGGL(up2_bwd_kernel, dim3(blocks_for(int64_t(N) * H * W * C)), dim3(256), 0, stream(), dout,
                       dout_stride, N, H, W, C, din, din_stride);
    SWP_LAUNCHED();
}

void pack_input(const float *const *src, const float *scale, int nsrc, int64_t P, uint16_t *x, int stride)
{
    SWP_CHECK(nsrc >= 1 && nsrc <= 4 && nsrc <= stride && x, "pack_input: bad arguments");
    Planes pl{};
    for (int c = 0; c < nsrc; ++c) {
        SWP_CHECK(src[c] != nullptr, "pack_input: null plane");
        pl.p[c] = src[c];
        pl.s[c] = scale[c];
    }
    hipLaunchKernelGGL(pack_input_kernel, dim3(blocks_for(P * stride)), dim3(256), 0, stream(), pl, nsrc, P, x,
                       stride);
    SWP_LAUNCHED();
}

void mse(const float *out, int out_stride, const float *target, const float *mask, int64_t P, double count,
         uint16_t *dout, int dout_stride, double *loss, double *partials)
{
    SWP_CHECK(out && target && dout && loss && partials && count > 0, "mse: bad arguments");
    const unsigned nb = unsigned(std::max<int64_t>(1, std::min<int64_t>((P + 1023) / 1024, 1024)));
    hipLaunchKernelGGL(mse_kernel, dim3(nb), dim3(256), 0, stream(), out, out_stride, target, mask, P, count, dout,
                       dout_stride, partials);
    SWP_LAUNCHED();
    hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(256), 0, stream(), partials, int(nb), 1.0 / count, loss);
    SWP_LAUNCHED();
}

void adam(float *w, const float *g, float *m, float *v, uint16_t *wbf, int64_t n, float lr, float b1, float b2,
          float eps, int step)
{
    SWP_CHECK(w && g && m && v && step >= 1, "adam: bad arguments");
    const float c1 = float(1.0 - std::pow(double(b1), step)), c2 = float(1.0 - std::pow(double(b2), step));
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(n)), dim3(256), 0, stream(), w, g, m, v, wbf, n, lr, b1, b2, eps,
                       c1, c2);
    SWP_LAUNCHED();
}

void to_bf16(const float *src, uint16_t *dst, int64_t n)
{
    SWP_CHECK(src && dst, "to_bf16: null buffer");
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n)), dim3(256), 0, stream(), src, dst, n);
    SWP_LAUNCHED();
}

}  // namespace nn
}  // namespace swp
