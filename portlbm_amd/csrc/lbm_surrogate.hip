// Warm-start surrogate: forward, backward and Adam kernels of a 14-conv
// encoder-decoder, and the executor that trains it on a device-resident
// dataset (include/lbm_surrogate.h).  FP32 throughout, FP64 only for the
// loss sums.  The network has no counterpart in the reference.
//
// Kernels (NCHW float32, 256-thread blocks):
//   k_conv3x3      implicit GEMM on the matrix cores, in FP32 or, for BF16
//                  inference, with BF16 operands; the input tile with its
//                  1-node halo staged in LDS; weights packed [Cout16][K16],
//                  K = 9 Cin in the weights' own (c, tap) order.  The data
//                  gradient is the same kernel on flipped, transposed weights.
//   k_conv_wgrad   the weight gradient on the same instruction, pixels as the
//                  inner dimension: a block has a 16 x 16 (out, in) channel
//                  pair and a slice of the pixel tiles; the slices' partial
//                  sums are added in a fixed order by k_wgrad_reduce, all
//                  convolutions in one launch.
//   pooling, upsampling, loss and Adam: one thread per element; the gradient
//   kernels that finish a layer's gradient apply its ReLU mask as they store.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "lbm_error.hpp"
#include "lbm_hip.h"
#include "lbm_surrogate.h"
#include "lbm_transfer.hpp"

namespace
{

constexpr int kConvs = LBM_SURROGATE_CONVS;
constexpr int kCin[kConvs] = {4, 16, 16, 32, 32, 48, 48, 64, 64, 64, 48, 32, 16, 16};
constexpr int kCout[kConvs] = {16, 16, 32, 32, 48, 48, 64, 64, 64, 48, 32, 16, 16, 3};

constexpr int kTile = 16;  // pixel tile edge of the weight gradient
constexpr int kWgT = 16;   // its channel tile

constexpr double kPi = 3.14159265358979323846;

inline int round16(int c) { return (c + 15) / 16 * 16; }

// Resolution level (0 = full, 4 = 1/16) at which conv k runs.
inline int conv_level(int k) { return k < 8 ? k / 2 : k == 8 ? 4 : k == 13 ? 0 : 12 - k; }

// ---- convolution on the matrix cores --------------------------------------
// y[b][o][p] = act(bias[o] + sum_k Wm[o][k] X[k][p]), k = c*9 + tap (the
// weights' own order), as an implicit GEMM in chunks of 16 k: in FP32 (E =
// float) four v_mfma_f32_16x16x4f32 per chunk, for BF16 inference (E = short)
// one v_mfma_f32_16x16x16bf16_1k, both with FP32 accumulation.
// Lane layouts, checked on the device.  BF16: A[i][k] in lane i + 16 (k/4),
// element k%4; B[k][j] in lane j + 16 (k/4), element k%4; D[i][j] in lane
// j + 16 (i/4), element i%4.  FP32: A[i][kk] in lane i + 16 kk, B[kk][j] in
// lane j + 16 kk, D as above; MFMA s of a chunk at kc gives slot kk the
// k = kc + 4 kk + s.  Either way a lane holds k = kc + 4 (lane/16) + 0..3 of
// both operands: its four weights are one load.
// A wave computes R rows of 16 pixels for CT tiles of 16 output channels: the
// rows share the weights, the tiles the pixels; four waves have 4 R rows, whose
// input with its 1-node halo is staged in LDS.
//
// The chunks are summed in the order of k (within a chunk, FP32 sums kc + s, kc +
// 4 + s, kc + 8 + s, kc + 12 + s for s = 0..3).  Another order moves activations across
// BF16 rounding bounds and across the zero of a ReLU, where the gradient jumps
// (taps before channels, with 16-byte LDS reads: no faster in FP32, and a
// gradient up to six times as far from FP64).  A lane's four pixels of a chunk
// so come from four places of the tile: their offsets are looked up in a table
// in LDS, once per chunk for the R rows.  Dividing per value instead, with one
// row per wave: 16 -> 16 channels at 256 x 256, BF16, 32 samples 242 us, here
// 97 us, bound by the 2-byte LDS reads; FP32, 16 samples 136 us, here 74 us (65
// TFLOP/s of 152 reachable; the 134 MB moved would take 27 us).  All
// convolutions of a BF16 prediction of 64 samples: 3.5 -> 1.7 ms, the 27 of a
// training batch of 16: 2.34 -> 1.4 ms.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kMfmaCols = 16;

__device__ __forceinline__ short f32_to_bf16_rne(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u)
        return short((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return short(u >> 16);
}

// A block's place (tile, sample) in a grid of (tiles, samples): the blocks that
// one XCD gets (every eighth in launch order) are neighbours, so that the
// halos and the lines that two tiles share are read into one L2.
__device__ __forceinline__ void xcd_place(unsigned &tile, unsigned &sample)
{
    const unsigned total = gridDim.x * gridDim.y, at = blockIdx.y * gridDim.x + blockIdx.x;
    const unsigned place = total % 8 == 0 ? (at % 8) * (total / 8) + at / 8 : at;
    tile = place % gridDim.x;
    sample = place / gridDim.x;
}

// relu: outputs below 0 become 0; mask (or null): outputs become 0 where it is
// not above 0 (the ReLU derivative of the layer below, for a data gradient).
// lo (or null): the input is x + up2(lo), lo of half the extents; a sum in
// memory of its own would be written and read once more (35 us for 16 channels
// at 256 x 256, 32 samples).
template <class E, int CT, int R>
__global__ __launch_bounds__(256) void k_conv3x3(const float *__restrict__ x, const float *__restrict__ lo,
                                                 const E *__restrict__ wm, const float *__restrict__ bias,
                                                 const float *__restrict__ mask, float *__restrict__ y, int Cin,
                                                 int Cout, int Kp, int H, int W, int tiles_x, int relu)
{
    typedef E E4 __attribute__((ext_vector_type(4)));
    constexpr bool kBf16 = sizeof(E) == 2;
    constexpr int TR = 4 * R + 2, TC = kMfmaCols + 2;
    extern __shared__ __align__(16) short conv_lds[];  // Kp offsets, then the tile and two channels of zeros
    short *offset = conv_lds;
    E *tile = reinterpret_cast<E *>(conv_lds + Kp);
    const int n = Cin * TR * TC;
    unsigned at, b;
    xcd_place(at, b);
    const int x0 = int(at % unsigned(tiles_x)) * kMfmaCols, y0 = int(at / unsigned(tiles_x)) * (4 * R);
    const float *xb = x + size_t(b) * Cin * H * W;
    for (int k = threadIdx.x; k < Kp; k += 256)
    {
        const int c = k / 9, tap = k - 9 * c;
        offset[k] = short((c * TR + tap / 3) * TC + tap % 3);  // below 66 * 18 * 18
    }
    // loads without branches, so that several are in flight
#pragma unroll 4
    for (int i = threadIdx.x; i < n; i += 256)
    {
        const int c = i / (TR * TC), px = i % (TR * TC);
        const int yy = y0 - 1 + px / TC, xx = x0 - 1 + px % TC;
        const bool in = yy >= 0 && yy < H && xx >= 0 && xx < W;
        float v = xb[in ? (size_t(c) * H + yy) * W + xx : 0];
        if (lo)
            v = lo[in ? ((size_t(b) * Cin + c) * (H / 2) + yy / 2) * (W / 2) + xx / 2 : 0] + v;
        v = in ? v : 0.f;
        if constexpr (kBf16)
            tile[i] = f32_to_bf16_rne(v);
        else
            tile[i] = v;
    }
    for (int i = n + threadIdx.x; i < n + 2 * TR * TC; i += 256)
        tile[i] = 0;  // the padding's k reach two channels past the last
    __syncthreads();
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int j = lane % 16, kq = 4 * (lane / 16);
    const int t0 = int(blockIdx.z) * CT;  // first tile of output channels
    f32x4 acc[CT][R];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int r = 0; r < R; ++r)
            acc[t][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    const E *xl = tile + wave * R * TC + j;
    const E *wl = wm + size_t(t0 * 16 + j) * Kp + kq;
    for (int kc = 0; kc < Kp; kc += 16)
    {
        const s16x4 from = *reinterpret_cast<const s16x4 *>(offset + kc + kq);
        E4 av[CT];
#pragma unroll
        for (int t = 0; t < CT; ++t)
            av[t] = *reinterpret_cast<const E4 *>(wl + size_t(t) * 16 * Kp + kc);
#pragma unroll
        for (int r = 0; r < R; ++r)
        {
            E4 bv;
#pragma unroll
            for (int it = 0; it < 4; ++it)
                bv[it] = xl[int(from[it]) + r * TC];
#pragma unroll
            for (int t = 0; t < CT; ++t)
            {
                if constexpr (kBf16)
                    acc[t][r] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[t], bv, acc[t][r], 0, 0, 0);
                else
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        acc[t][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[t][s], bv[s], acc[t][r], 0, 0, 0);
            }
        }
    }
    const int ox = x0 + j;
#pragma unroll
    for (int r = 0; r < R; ++r)
    {
        const int oy = y0 + wave * R + r;
        if (oy >= H || ox >= W)
            continue;
#pragma unroll
        for (int t = 0; t < CT; ++t)
        {
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int co = (t0 + t) * 16 + kq + v;
                if (co < Cout)
                {
                    const size_t to = ((size_t(b) * Cout + co) * H + oy) * W + ox;
                    float o = acc[t][r][v] + (bias ? bias[co] : 0.f);
                    if (relu)
                        o = o > 0.f ? o : 0.f;
                    if (mask && !(mask[to] > 0.f))
                        o = 0.f;
                    y[to] = o;
                }
            }
        }
    }
}

// Partial weight/bias gradient of one slice of (sample, tile) pairs:
// partial[((slice*CoutP + o)*CinP + c)*10 + k] = sum g[b,o,i,j] x[b,c,i+ky-1,j+kx-1] (k < 9),
// slot 9 = sum g[b,o,i,j].  Per 16-pixel row of a tile and tap, four
// v_mfma_f32_16x16x4f32 with A = g (16 output channels x 4 pixels) and B = x
// (4 pixels x 16 input channels); slot kk of MFMA s is pixel 4 kk + s.  A
// lane's six pixels of an input row serve the three taps of that row.  A wave
// takes four rows of the tile; the four waves' sums are added in wave order.
// The strides put the 16 channels of a read on different banks.
//
// Bound by the staging: the loads of a tile are all issued before the barrier
// that ends the tile before it.  16 x 16 channels, 16 samples of 256 x 256: 70
// us; 96 us with a loop of guarded loads.  All convolutions of that batch with
// their reductions: 1.38 ms with one thread per channel pair (no matrix unit,
// four times the slices, two reduction launches each), 0.65 ms this way.
constexpr int kGStride = kTile * kTile + 4;
constexpr int kXRow = kTile + 4, kXStride = (kTile + 2) * kXRow + 4;

__global__ __launch_bounds__(256) void k_conv_wgrad(const float *__restrict__ x, const float *__restrict__ lo,
                                                    const float *__restrict__ g, float *__restrict__ partial, int B,
                                                    int Cin, int Cout, int CinP, int CoutP, int H, int W, int tiles_x,
                                                    int tiles_per_image, int slices)
{
    __shared__ __align__(16) float lds[kWgT * (kGStride + kXStride)];
    float *gs = lds, *xs = lds + kWgT * kGStride;
    static_assert(3 * 9 * 256 + 3 * 64 <= kWgT * (kGStride + kXStride), "the waves' sums fit");
    const int ci_tiles = CinP / kWgT;
    const int co0 = int(blockIdx.x / unsigned(ci_tiles)) * kWgT, ci0 = int(blockIdx.x % unsigned(ci_tiles)) * kWgT;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, ch = lane % 16, kk = 4 * (lane / 16);
    f32x4 acc[9];
#pragma unroll
    for (int k = 0; k < 9; ++k)
        acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.f;
    const int total = B * tiles_per_image;
    for (int t = blockIdx.y; t < total; t += slices)
    {
        const int b = t / tiles_per_image, tt = t % tiles_per_image;
        const int tx0 = (tt % tiles_x) * kTile, ty0 = (tt / tiles_x) * kTile;
        // Sixteen threads per channel, one per column: every load of a thread
        // is a fixed number of rows from its first, and none waits for
        // another; the columns left and right of the tile come last.
        const int c = threadIdx.x / kTile, col = threadIdx.x % kTile;
        const float *gc = g + (size_t(b) * Cout + min(co0 + c, Cout - 1)) * H * W;
        const float *xc = x + (size_t(b) * Cin + min(ci0 + c, Cin - 1)) * H * W;
        const bool gin = co0 + c < Cout && tx0 + col < W, xin = ci0 + c < Cin;
        float gv[kTile], xv[kTile + 2], ev[3];
#pragma unroll
        for (int r = 0; r < kTile; ++r)
        {
            const bool in = gin && ty0 + r < H;
            gv[r] = gc[in ? (ty0 + r) * W + tx0 + col : 0];
            gv[r] = in ? gv[r] : 0.f;
        }
#pragma unroll
        for (int r = 0; r < kTile + 2; ++r)
        {
            const int yy = ty0 + r - 1;
            const bool in = xin && tx0 + col < W && yy >= 0 && yy < H;
            xv[r] = xc[in ? yy * W + tx0 + col : 0];
            xv[r] = in ? xv[r] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 3; ++e)
        {
            const int i = col + e * kTile, yy = ty0 + i / 2 - 1, xx = tx0 + (i % 2 ? kTile : -1);
            const bool in = xin && i < 2 * (kTile + 2) && xx >= 0 && xx < W && yy >= 0 && yy < H;
            ev[e] = xc[in ? yy * W + xx : 0];
            ev[e] = in ? ev[e] : 0.f;
        }
        if (lo)  // the input is x + up2(lo)
        {
            const float *lc = lo + (size_t(b) * Cin + min(ci0 + c, Cin - 1)) * (H / 2) * (W / 2);
            float lv[kTile / 2 + 2], le[3];
#pragma unroll
            for (int r = 0; r < kTile / 2 + 2; ++r)  // rows 2 r - 1 and 2 r of the tile with its halo
            {
                const int yy = ty0 / 2 + r - 1;
                const bool in = xin && tx0 + col < W && yy >= 0 && yy < H / 2;
                lv[r] = lc[in ? yy * (W / 2) + (tx0 + col) / 2 : 0];
                lv[r] = in ? lv[r] : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 3; ++e)
            {
                const int i = col + e * kTile, yy = ty0 + i / 2 - 1, xx = tx0 + (i % 2 ? kTile : -1);
                const bool in = xin && i < 2 * (kTile + 2) && xx >= 0 && xx < W && yy >= 0 && yy < H;
                le[e] = lc[in ? yy / 2 * (W / 2) + xx / 2 : 0];
                ev[e] += in ? le[e] : 0.f;
            }
#pragma unroll
            for (int r = 0; r < kTile + 2; ++r)
                xv[r] += lv[(r + 1) / 2];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kTile; ++r)
            gs[c * kGStride + r * kTile + col] = gv[r];
#pragma unroll
        for (int r = 0; r < kTile + 2; ++r)
            xs[c * kXStride + r * kXRow + 1 + col] = xv[r];
#pragma unroll
        for (int e = 0; e < 3; ++e)
        {
            const int i = col + e * kTile;
            if (i < 2 * (kTile + 2))
                xs[c * kXStride + i / 2 * kXRow + (i % 2 ? kTile + 1 : 0)] = ev[e];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            const int r = 4 * wave + q;
            const f32x4 a = *reinterpret_cast<const f32x4 *>(gs + ch * kGStride + r * kTile + kk);
            bsum += ((a[0] + a[1]) + a[2]) + a[3];
#pragma unroll
            for (int ky = 0; ky < 3; ++ky)
            {
                const float *xr = xs + ch * kXStride + (r + ky) * kXRow + kk;
                const f32x4 lo = *reinterpret_cast<const f32x4 *>(xr);
                const float v[6] = {lo[0], lo[1], lo[2], lo[3], xr[4], xr[5]};
#pragma unroll
                for (int kx = 0; kx < 3; ++kx)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        acc[3 * ky + kx] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], v[s + kx], acc[3 * ky + kx], 0, 0, 0);
            }
        }
    }
    // D[i][j]: output channel 4 (lane / 16) + v, input channel lane % 16
    __syncthreads();
    bsum += __shfl_xor(bsum, 16, 64);
    bsum += __shfl_xor(bsum, 32, 64);  // every lane: its channel's (lane % 16) sum
    if (wave > 0)
    {
#pragma unroll
        for (int k = 0; k < 9; ++k)
            *reinterpret_cast<f32x4 *>(lds + (((wave - 1) * 9 + k) * 64 + lane) * 4) = acc[k];
        lds[3 * 9 * 256 + (wave - 1) * 64 + lane] = bsum;
    }
    __syncthreads();
    if (wave > 0)
        return;
    for (int w = 0; w < 3; ++w)
    {
#pragma unroll
        for (int k = 0; k < 9; ++k)
            acc[k] += *reinterpret_cast<const f32x4 *>(lds + ((w * 9 + k) * 64 + lane) * 4);
        bsum += lds[3 * 9 * 256 + w * 64 + lane];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
    {
        float *out = partial + ((size_t(blockIdx.y) * CoutP + co0 + kk + v) * CinP + ci0 + ch) * 10;
#pragma unroll
        for (int k = 0; k < 9; ++k)
            out[k] = acc[k][v];
    }
    if (lane < 16)
        partial[((size_t(blockIdx.y) * CoutP + co0 + ch) * CinP + ci0) * 10 + 9] = bsum;
}

// The gradients of every convolution from the slices' partial sums, in one
// launch and a fixed order (bitwise reproducible, FP64): a block has 32
// weights of one convolution, eight threads each take every eighth slice, and
// their sums are added in order.  Weight index w < Cout*Cin*9 is (o, c, k),
// then Cout biases (slot 9 of channel 0).
constexpr int kReduceWeights = 32, kReduceGroups = 8;

struct ReduceConv
{
    const float *partial;
    float *grad;  // weights, then biases
    int Cin, Cout, CinP, CoutP, slices;
    int first_block;
};
struct ReduceAll
{
    ReduceConv conv[kConvs];
};

__global__ __launch_bounds__(kReduceWeights *kReduceGroups) void k_wgrad_reduce(ReduceAll a)
{
    int k = 0;
    while (k + 1 < kConvs && int(blockIdx.x) >= a.conv[k + 1].first_block)
        ++k;
    const ReduceConv cv = a.conv[k];
    const int wl = threadIdx.x % kReduceWeights, group = threadIdx.x / kReduceWeights;
    const int w = (int(blockIdx.x) - cv.first_block) * kReduceWeights + wl;
    const int nw = cv.Cout * cv.Cin * 9, nall = nw + cv.Cout;
    double sum = 0.0;
    if (w < nall)
    {
        const int o = w < nw ? w / (cv.Cin * 9) : w - nw, c = w < nw ? (w / 9) % cv.Cin : 0;
        const size_t slot = (size_t(o) * cv.CinP + c) * 10 + (w < nw ? w % 9 : 9);
        const size_t stride = size_t(cv.CoutP) * cv.CinP * 10;
#pragma unroll 8
        for (int s = group; s < cv.slices; s += kReduceGroups)
            sum += double(cv.partial[size_t(s) * stride + slot]);
    }
    __shared__ double part[kReduceGroups][kReduceWeights];
    part[group][wl] = sum;
    __syncthreads();
    if (group == 0 && w < nall)
    {
        for (int g = 1; g < kReduceGroups; ++g)
            sum += part[g][wl];
        cv.grad[w] = float(sum);
    }
}

// wb[o*Kp + k] = bf16(w[o*9Cin + k]) for k < 9 Cin (padding stays zero)
__global__ void k_pack_bf16(const float *__restrict__ w, short *__restrict__ wb, int Cin, int Cout, int Kp)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const int K = 9 * Cin;
    if (idx >= Cout * K)
        return;
    const int o = idx / K, k = idx % K;
    wb[size_t(o) * Kp + k] = f32_to_bf16_rne(w[idx]);
}

// wm[o*Kp + c*9 + k] = w[o][c][k] (Kp = round16(9 Cin));
// wt[c*KpT + o*9 + 8-k] = w[o][c][k] (KpT = round16(9 Cout)): the data
// gradient's weights, input and output channels swapped, taps flipped.
// Padding rows and columns stay zero.
__global__ void k_pack(const float *__restrict__ w, float *__restrict__ wm, float *__restrict__ wt, int Cin, int Cout,
                       int Kp, int KpT)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= Cout * Cin * 9)
        return;
    const int o = idx / (Cin * 9), c = (idx / 9) % Cin, k = idx % 9;
    wm[size_t(o) * Kp + c * 9 + k] = w[idx];
    wt[size_t(c) * KpT + o * 9 + (8 - k)] = w[idx];
}

__global__ void k_pool2(const float *__restrict__ x, float *__restrict__ y, int BC, int H, int W)
{
    const int h = H / 2, w = W / 2;
    const size_t n = size_t(BC) * h * w;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    {
        const size_t bc = i / (size_t(h) * w);
        const int r = int(i % (size_t(h) * w)), yi = r / w, xi = r % w;
        const float *p = x + (bc * H + 2 * yi) * W + 2 * xi;
        y[i] = 0.25f * (((p[0] + p[1]) + p[W]) + p[W + 1]);
    }
}

// dx[b,c,y,x] = [a > 0] (dx + 0.25 dy[b,c,y/2,x/2]): the last share of the
// gradient of a, with its ReLU mask
__global__ void k_pool2_backward_add(const float *__restrict__ dy, const float *__restrict__ a,
                                     float *__restrict__ dx, int BC, int H, int W)
{
    const size_t n = size_t(BC) * H * W;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    {
        const size_t bc = i / (size_t(H) * W);
        const int r = int(i % (size_t(H) * W)), yi = r / W, xi = r % W;
        const float v = dx[i] + 0.25f * dy[(bc * (H / 2) + yi / 2) * (W / 2) + xi / 2];
        dx[i] = a[i] > 0.f ? v : 0.f;
    }
}

// dlo[b,c,i,j] = [a > 0] (sum of dz over the 2x2 block) (dlo, a: H/2 x W/2)
__global__ void k_upsample_backward(const float *__restrict__ dz, const float *__restrict__ a,
                                    float *__restrict__ dlo, int BC, int H, int W)
{
    const int h = H / 2, w = W / 2;
    const size_t n = size_t(BC) * h * w;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    {
        const size_t bc = i / (size_t(h) * w);
        const int r = int(i % (size_t(h) * w)), yi = r / w, xi = r % w;
        const float *p = dz + (bc * H + 2 * yi) * W + 2 * xi;
        dlo[i] = a[i] > 0.f ? ((p[0] + p[1]) + p[W]) + p[W + 1] : 0.f;
    }
}

constexpr int kLossBlocks = 2048;  // at most

// dout = 2 m (out - t) norm; partial[block] = sum m (out - t)^2 (FP64)
__global__ __launch_bounds__(256) void k_loss(const float *__restrict__ out, const float *__restrict__ tgt,
                                              const float *__restrict__ in, float *__restrict__ dout,
                                              double *__restrict__ partial, int B, int HW, float norm)
{
    const size_t n = size_t(B) * LBM_SURROGATE_OUTPUTS * HW;
    double s = 0.0;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    {
        const size_t b = i / (size_t(LBM_SURROGATE_OUTPUTS) * HW);
        const size_t p = i % size_t(HW);
        const float m = in[b * LBM_SURROGATE_INPUTS * size_t(HW) + p];
        const float e = out[i] - tgt[i];
        s += double(m) * double(e) * double(e);
        dout[i] = 2.f * m * e * norm;
    }
    __shared__ double part[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0)
        partial[blockIdx.x] = ((part[0] + part[1]) + part[2]) + part[3];
}

// partial[block] = sum of the fluid masks of B samples (FP64; exact for a mask of
// zeros and ones).  With the host's serial sum of that million floats a gradient
// of 16 samples of 256 x 256 took 3.81 ms, with this 3.39.
__global__ __launch_bounds__(256) void k_mask_sum(const float *__restrict__ in, double *__restrict__ partial, int B,
                                                  int HW)
{
    const size_t n = size_t(B) * HW;
    double s = 0.0;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
        s += double(in[i / size_t(HW) * LBM_SURROGATE_INPUTS * size_t(HW) + i % size_t(HW)]);
    __shared__ double part[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0)
        partial[blockIdx.x] = ((part[0] + part[1]) + part[2]) + part[3];
}

// the blocks' sums in a fixed order: a thread's every 256th, then the threads'
__global__ __launch_bounds__(256) void k_loss_final(const double *__restrict__ partial, int blocks, double norm,
                                                    double *__restrict__ loss, float *__restrict__ history, int slot)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < blocks; i += 256)
        s += partial[i];
    __shared__ double part[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    s = (((part[0] + part[1]) + part[2]) + part[3]) * norm;
    *loss = s;
    if (history)
        history[slot] = float(s);
}

// Adam step (bias-corrected): c1 = 1 - b1^t, c2 = 1 - b2^t
__global__ void k_adam(float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
                       const float *__restrict__ g, size_t n, float lr, float b1, float b2, float eps, float c1,
                       float c2)
{
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

inline unsigned elem_grid(size_t n) { return unsigned(std::min<size_t>((n + 255) / 256, 8192)); }

uint64_t splitmix64(uint64_t &state)
{
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

double uniform01(uint64_t &state) { return double(splitmix64(state) >> 11) * 0x1.0p-53; }

#define S_TRY(expr)                                                                                    \
    do                                                                                                 \
    {                                                                                                  \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return lbm_set_error(e_ == hipErrorOutOfMemory ? LBM_ERR_OUT_OF_MEMORY : LBM_ERR_DEVICE,   \
                                 std::string(#expr) + ": " + hipGetErrorString(e_));                  \
    } while (0)

}  // namespace

struct lbm_surrogate
{
    int H = 0, W = 0, Bmax = 0;
    int LH[5] = {}, LW[5] = {};
    size_t nparams = 0;
    size_t w_off[kConvs] = {}, b_off[kConvs] = {};
    float *params = nullptr, *grad = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    float *wp[kConvs] = {}, *wt[kConvs] = {};
    short *wb[kConvs] = {};  // BF16 [Cout16][K16] weights of the matrix-core inference
    bool packed = false;
    uint32_t adam_t = 0;
    float *in = nullptr, *tgt = nullptr, *out = nullptr, *dout = nullptr, *dtmp = nullptr;
    float *a[14] = {}, *p[5] = {}, *da[14] = {};
    float *partial[kConvs] = {};  // the weight gradients' slices
    double *loss_part = nullptr, *loss_dev = nullptr;  // loss_dev: the loss, a mask sum
    float *history = nullptr;
    size_t history_cap = 0;
    float *ds_in = nullptr, *ds_tgt = nullptr;
    size_t ds_cap = 0, ds_n = 0;
    std::vector<double> ds_fluid;
    // training schedule and shuffle state, carried across train calls
    uint32_t sched_step = 0;
    bool shuffle_seeded = false;
    uint64_t shuffle_state = 0;
    std::vector<uint32_t> perm;
    size_t cursor = 0;
    std::vector<void *> allocations;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_ms = 0.0;
};

namespace
{

size_t param_count()
{
    size_t n = 0;
    for (int k = 0; k < kConvs; ++k)
        n += size_t(kCout[k]) * kCin[k] * 9 + kCout[k];
    return n;
}

int alloc(lbm_surrogate *s, float **ptr, size_t floats)
{
    void *v = nullptr;
    S_TRY(hipMalloc(&v, std::max<size_t>(floats, 1) * sizeof(float)));
    s->allocations.push_back(v);
    *ptr = static_cast<float *>(v);
    return LBM_OK;
}

size_t act_floats(const lbm_surrogate *s, int C, int level)
{
    return size_t(s->Bmax) * C * s->LH[level] * s->LW[level];
}

int tiles_x(const lbm_surrogate *s, int l) { return (s->LW[l] + kTile - 1) / kTile; }
int tiles(const lbm_surrogate *s, int l) { return tiles_x(s, l) * ((s->LH[l] + kTile - 1) / kTile); }

// Weight-gradient slices: the blocks that fit the GPU at once (four per compute
// unit by their LDS), at most one tile each.  Half as many took 140 instead of
// 96 us for 16 x 16 channels at 256 x 256, 16 samples.
int wgrad_slices(const lbm_surrogate *s, int k, int l, int B)
{
    const int blocks = (round16(kCout[k]) / kWgT) * (round16(kCin[k]) / kWgT);
    return std::min(std::max(1, 1024 / blocks), B * tiles(s, l));
}

int pack_all(lbm_surrogate *s)
{
    for (int k = 0; k < kConvs; ++k)
    {
        const int n = kCout[k] * kCin[k] * 9;
        hipLaunchKernelGGL(k_pack, dim3((n + 255) / 256), dim3(256), 0, s->stream, s->params + s->w_off[k], s->wp[k],
                           s->wt[k], kCin[k], kCout[k], round16(9 * kCin[k]), round16(9 * kCout[k]));
        hipLaunchKernelGGL(k_pack_bf16, dim3((n + 255) / 256), dim3(256), 0, s->stream, s->params + s->w_off[k],
                           s->wb[k], kCin[k], kCout[k], round16(9 * kCin[k]));
    }
    S_TRY(hipGetLastError());
    s->packed = true;
    return LBM_OK;
}

// Calls f(CT, R) with the output-channel tiles per block and the rows per wave
// of a convolution.  Rows of a wave share the weights and most of the halo,
// channel tiles share the staged input: four rows and all channel tiles where
// that leaves two blocks per compute unit (512), two rows, then one row below
// that (two at most for more than 32 input channels, in either type: 48 in FP32
// would take 65.7 KB, above the 64 KB that a launch gets unasked); the channel
// tiles of a layer too small for 512 blocks of one row get blocks of their own.
// 16 -> 16 channels at 256 x 256, 16 samples in FP32: 136 us with one row, 74 us
// with four.
template <class F>
void conv_shape(int Cin, int Cout, int H, int W, int B, F f)
{
    using std::integral_constant;
    const int co_tiles = (Cout + 15) / 16, cols = (W + kMfmaCols - 1) / kMfmaCols;
    auto blocks = [&](int rows) { return size_t(cols) * ((H + 4 * rows - 1) / (4 * rows)) * B; };
    auto by_rows = [&](auto ct) {
        if (Cin <= 32 && blocks(4) * (co_tiles / ct.value) >= 512)
            f(ct, integral_constant<int, 4>{});
        else if (blocks(2) * (co_tiles / ct.value) >= 512)
            f(ct, integral_constant<int, 2>{});
        else
            f(ct, integral_constant<int, 1>{});
    };
    if (co_tiles > 1 && blocks(1) < 512)
        by_rows(integral_constant<int, 1>{});
    else if (co_tiles == 1)
        by_rows(integral_constant<int, 1>{});
    else if (co_tiles == 2)
        by_rows(integral_constant<int, 2>{});
    else if (co_tiles == 3)
        by_rows(integral_constant<int, 3>{});
    else
        by_rows(integral_constant<int, 4>{});
}

// Convolution of x, or of x + up2(lo), with packed weights wm ([Cout16][round16(9 Cin)]) into y.
template <class E>
void conv(lbm_surrogate *s, const float *x, const float *lo, const E *wm, const float *bias, const float *mask,
          float *y, int Cin, int Cout, int l, int B, bool relu)
{
    const int H = s->LH[l], W = s->LW[l], tx = (W + kMfmaCols - 1) / kMfmaCols, Kp = round16(9 * Cin);
    conv_shape(Cin, Cout, H, W, B, [&](auto ct, auto rows) {
        constexpr int CT = decltype(ct)::value, R = decltype(rows)::value;
        const int ty = (H + 4 * R - 1) / (4 * R);
        const size_t lds = size_t(Cin + 2) * (4 * R + 2) * (kMfmaCols + 2) * sizeof(E) + size_t(Kp) * sizeof(short);
        const dim3 grid(unsigned(tx * ty), unsigned(B), unsigned((Cout + 15) / 16 / CT));
        hipLaunchKernelGGL((k_conv3x3<E, CT, R>), grid, dim3(256), lds, s->stream, x, lo, wm, bias, mask, y, Cin, Cout,
                           Kp, H, W, tx, relu ? 1 : 0);
    });
}

void conv_forward(lbm_surrogate *s, const float *x, const float *lo, int k, float *y, int l, int B, bool relu,
                  bool bf16)
{
    const float *bias = s->params + s->b_off[k];
    if (bf16)
        conv<short>(s, x, lo, s->wb[k], bias, nullptr, y, kCin[k], kCout[k], l, B, relu);
    else
        conv<float>(s, x, lo, s->wp[k], bias, nullptr, y, kCin[k], kCout[k], l, B, relu);
}

// dx = data gradient of conv k for output gradient g (dx written, not
// accumulated), with the ReLU mask of activation a (null: none)
void conv_dgrad(lbm_surrogate *s, const float *g, int k, const float *a, float *dx, int l, int B)
{
    conv<float>(s, g, nullptr, s->wt[k], nullptr, a, dx, kCout[k], kCin[k], l, B, false);
}

void conv_wgrad(lbm_surrogate *s, const float *x, const float *lo, const float *g, int k, int l, int B)
{
    const int CinP = round16(kCin[k]), CoutP = round16(kCout[k]);
    const int slices = wgrad_slices(s, k, l, B);
    const dim3 grid(unsigned((CoutP / kWgT) * (CinP / kWgT)), unsigned(slices));
    hipLaunchKernelGGL(k_conv_wgrad, grid, dim3(256), 0, s->stream, x, lo, g, s->partial[k], B, kCin[k], kCout[k],
                       CinP, CoutP, s->LH[l], s->LW[l], tiles_x(s, l), tiles(s, l), slices);
}

// every convolution's gradient from its slices
void wgrad_reduce(lbm_surrogate *s, int B)
{
    ReduceAll a{};
    int blocks = 0;
    for (int k = 0; k < kConvs; ++k)
    {
        a.conv[k] = ReduceConv{s->partial[k],        s->grad + s->w_off[k],
                               kCin[k],              kCout[k],
                               round16(kCin[k]),     round16(kCout[k]),
                               wgrad_slices(s, k, conv_level(k), B), blocks};
        blocks += (kCout[k] * kCin[k] * 9 + kCout[k] + kReduceWeights - 1) / kReduceWeights;
    }
    hipLaunchKernelGGL(k_wgrad_reduce, dim3(unsigned(blocks)), dim3(kReduceWeights * kReduceGroups), 0, s->stream, a);
}

void pool(lbm_surrogate *s, const float *x, float *y, int C, int l_in, int B)
{
    const size_t n = size_t(B) * C * s->LH[l_in + 1] * s->LW[l_in + 1];
    hipLaunchKernelGGL(k_pool2, dim3(elem_grid(n)), dim3(256), 0, s->stream, x, y, B * C, s->LH[l_in], s->LW[l_in]);
}

void pool_backward_add(lbm_surrogate *s, const float *dy, const float *a, float *dx, int C, int l_in, int B)
{
    const size_t n = size_t(B) * C * s->LH[l_in] * s->LW[l_in];
    hipLaunchKernelGGL(k_pool2_backward_add, dim3(elem_grid(n)), dim3(256), 0, s->stream, dy, a, dx, B * C,
                       s->LH[l_in], s->LW[l_in]);
}

void upsample_backward(lbm_surrogate *s, const float *dz, const float *a, float *dlo, int C, int l, int B)
{
    const size_t n = size_t(B) * C * s->LH[l + 1] * s->LW[l + 1];
    hipLaunchKernelGGL(k_upsample_backward, dim3(elem_grid(n)), dim3(256), 0, s->stream, dz, a, dlo, B * C, s->LH[l],
                       s->LW[l]);
}

// Forward over s->in (B samples) into s->a, s->p, s->out; bf16: the
// convolutions on the matrix cores (inference).
void forward(lbm_surrogate *s, int B, bool bf16 = false)
{
    conv_forward(s, s->in, nullptr, 0, s->a[1], 0, B, true, bf16);
    conv_forward(s, s->a[1], nullptr, 1, s->a[2], 0, B, true, bf16);
    for (int l = 1; l <= 3; ++l)
    {
        pool(s, s->a[2 * l], s->p[l], kCout[2 * l - 1], l - 1, B);
        conv_forward(s, s->p[l], nullptr, 2 * l, s->a[2 * l + 1], l, B, true, bf16);
        conv_forward(s, s->a[2 * l + 1], nullptr, 2 * l + 1, s->a[2 * l + 2], l, B, true, bf16);
    }
    pool(s, s->a[8], s->p[4], kCout[7], 3, B);
    conv_forward(s, s->p[4], nullptr, 8, s->a[9], 4, B, true, bf16);
    for (int m = 0; m < 4; ++m)
    {
        const int l = 3 - m, kk = 9 + m;
        conv_forward(s, s->a[8 - 2 * m], s->a[9 + m], kk, s->a[10 + m], l, B, true, bf16);
    }
    conv_forward(s, s->a[13], nullptr, 13, s->out, 0, B, false, bf16);
}

// Loss of s->out against s->tgt and the full parameter gradient into s->grad.
void loss_backward(lbm_surrogate *s, int B, double norm, float *history, int slot)
{
    const int HW = s->H * s->W;
    const unsigned blocks =
        std::min<unsigned>(kLossBlocks, elem_grid(size_t(B) * LBM_SURROGATE_OUTPUTS * size_t(HW)));
    hipLaunchKernelGGL(k_loss, dim3(blocks), dim3(256), 0, s->stream, s->out, s->tgt, s->in, s->dout, s->loss_part, B,
                       HW, float(norm));
    hipLaunchKernelGGL(k_loss_final, dim3(1), dim3(256), 0, s->stream, s->loss_part, int(blocks), norm, s->loss_dev,
                       history, slot);
    // Every da[] is complete, ReLU mask included, once its last share is in.
    // conv13 (no ReLU)
    conv_wgrad(s, s->a[13], nullptr, s->dout, 13, 0, B);
    conv_dgrad(s, s->dout, 13, s->a[13], s->da[13], 0, B);
    for (int m = 3; m >= 0; --m)
    {
        const int l = 3 - m, kk = 9 + m;
        conv_wgrad(s, s->a[8 - 2 * m], s->a[9 + m], s->da[10 + m], kk, l, B);
        // the gradient of the sum is the skip's: written straight into da[8-2m], which
        // the pool's share completes
        conv_dgrad(s, s->da[10 + m], kk, nullptr, s->da[8 - 2 * m], l, B);
        upsample_backward(s, s->da[8 - 2 * m], s->a[9 + m], s->da[9 + m], kCin[kk], l, B);
    }
    conv_wgrad(s, s->p[4], nullptr, s->da[9], 8, 4, B);
    conv_dgrad(s, s->da[9], 8, nullptr, s->dtmp, 4, B);
    pool_backward_add(s, s->dtmp, s->a[8], s->da[8], kCin[8], 3, B);
    for (int l = 3; l >= 0; --l)
    {
        const int k1 = 2 * l + 1, k0 = 2 * l;
        conv_wgrad(s, s->a[k1], nullptr, s->da[k1 + 1], k1, l, B);
        conv_dgrad(s, s->da[k1 + 1], k1, s->a[k1], s->da[k1], l, B);
        conv_wgrad(s, l == 0 ? s->in : s->p[l], nullptr, s->da[k1], k0, l, B);
        if (l > 0)
        {
            conv_dgrad(s, s->da[k1], k0, nullptr, s->dtmp, l, B);
            pool_backward_add(s, s->dtmp, s->a[k0], s->da[k0], kCin[k0], l - 1, B);
        }
    }
    wgrad_reduce(s, B);
}

int adam_step(lbm_surrogate *s, float lr)
{
    const double b1 = 0.9, b2 = 0.999;
    ++s->adam_t;
    const double c1 = 1.0 - std::pow(b1, double(s->adam_t)), c2 = 1.0 - std::pow(b2, double(s->adam_t));
    hipLaunchKernelGGL(k_adam, dim3(elem_grid(s->nparams)), dim3(256), 0, s->stream, s->params, s->adam_m, s->adam_v,
                       s->grad, s->nparams, lr, float(b1), float(b2), 1e-8f, float(c1), float(c2));
    S_TRY(hipGetLastError());
    return pack_all(s);
}

int reset_adam(lbm_surrogate *s)
{
    s->sched_step = 0;
    s->shuffle_seeded = false;
    S_TRY(hipMemsetAsync(s->adam_m, 0, s->nparams * sizeof(float), s->stream));
    S_TRY(hipMemsetAsync(s->adam_v, 0, s->nparams * sizeof(float), s->stream));
    s->adam_t = 0;
    return LBM_OK;
}

double fluid_sum(const float *inputs, uint32_t batch, size_t hw)
{
    double m = 0.0;
    for (uint32_t b = 0; b < batch; ++b)
    {
        const float *c0 = inputs + size_t(b) * LBM_SURROGATE_INPUTS * hw;
        for (size_t i = 0; i < hw; ++i)
            m += double(c0[i]);
    }
    return m;
}

int check_ready(const lbm_surrogate *s, const char *what)
{
    if (!s)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, std::string(what) + ": null handle");
    if (!s->packed)
        return lbm_set_error(LBM_ERR_STATE, std::string(what) + ": parameters not set (init or set them first)");
    return LBM_OK;
}

}  // namespace

extern "C" {

size_t lbm_surrogate_param_count(void) { return param_count(); }

void lbm_surrogate_destroy(lbm_surrogate *s)
{
    if (!s)
        return;
    if (s->stream)
        (void)hipStreamSynchronize(s->stream);
    for (void *v : s->allocations)
        (void)hipFree(v);
    (void)hipFree(s->loss_part);
    (void)hipFree(s->loss_dev);
    (void)hipFree(s->history);
    (void)hipFree(s->ds_in);
    (void)hipFree(s->ds_tgt);
    if (s->ev0)
        (void)hipEventDestroy(s->ev0);
    if (s->ev1)
        (void)hipEventDestroy(s->ev1);
    if (s->stream)
        (void)hipStreamDestroy(s->stream);
    delete s;
}

int lbm_surrogate_create(uint32_t height, uint32_t width, uint32_t max_batch, lbm_surrogate **out)
{
    if (!out)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_create: null output");
    *out = nullptr;
    if (height == 0 || width == 0 || height % 16 || width % 16 || height > 8192 || width > 8192 || max_batch == 0 ||
        max_batch > 4096)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT,
                             "lbm_surrogate_create: height and width must be positive multiples of 16 (<= 8192), "
                             "max_batch in 1..4096");
    auto *s = new lbm_surrogate;
    s->H = int(height);
    s->W = int(width);
    s->Bmax = int(max_batch);
    for (int l = 0; l < 5; ++l)
    {
        s->LH[l] = s->H >> l;
        s->LW[l] = s->W >> l;
    }
    size_t off = 0;
    for (int k = 0; k < kConvs; ++k)
    {
        s->w_off[k] = off;
        off += size_t(kCout[k]) * kCin[k] * 9;
        s->b_off[k] = off;
        off += kCout[k];
    }
    s->nparams = off;
    int rc = LBM_OK;
#define C_TRY(expr)                                                                                    \
    do                                                                                                 \
    {                                                                                                  \
        if ((rc = (expr)) != LBM_OK)                                                                   \
        {                                                                                              \
            lbm_surrogate_destroy(s);                                                                  \
            return rc;                                                                                 \
        }                                                                                              \
    } while (0)
    C_TRY([&]() -> int {
        S_TRY(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
        S_TRY(hipEventCreate(&s->ev0));
        S_TRY(hipEventCreate(&s->ev1));
        S_TRY(hipMalloc(&s->loss_part, kLossBlocks * sizeof(double)));
        S_TRY(hipMalloc(&s->loss_dev, 2 * sizeof(double)));
        return LBM_OK;
    }());
    C_TRY(alloc(s, &s->params, s->nparams));
    C_TRY(alloc(s, &s->grad, s->nparams));
    C_TRY(alloc(s, &s->adam_m, s->nparams));
    C_TRY(alloc(s, &s->adam_v, s->nparams));
    for (int k = 0; k < kConvs; ++k)
    {
        const size_t cin_p = size_t(round16(kCin[k])), cout_p = size_t(round16(kCout[k]));
        C_TRY(alloc(s, &s->wp[k], cin_p * 9 * cout_p));
        C_TRY(alloc(s, &s->wt[k], cin_p * 9 * cout_p));
        const size_t kp = size_t(round16(9 * kCin[k]));
        float *wbf = nullptr;
        C_TRY(alloc(s, &wbf, (cout_p * kp + 1) / 2));
        s->wb[k] = reinterpret_cast<short *>(wbf);
        C_TRY([&]() -> int {
            S_TRY(hipMemsetAsync(s->wp[k], 0, cin_p * 9 * cout_p * sizeof(float), s->stream));
            S_TRY(hipMemsetAsync(s->wt[k], 0, cin_p * 9 * cout_p * sizeof(float), s->stream));
            S_TRY(hipMemsetAsync(s->wb[k], 0, cout_p * kp * sizeof(short), s->stream));
            return LBM_OK;
        }());
        C_TRY(alloc(s, &s->partial[k], size_t(wgrad_slices(s, k, conv_level(k), s->Bmax)) * cout_p * cin_p * 10));
    }
    C_TRY(alloc(s, &s->in, act_floats(s, LBM_SURROGATE_INPUTS, 0)));
    C_TRY(alloc(s, &s->tgt, act_floats(s, LBM_SURROGATE_OUTPUTS, 0)));
    C_TRY(alloc(s, &s->out, act_floats(s, LBM_SURROGATE_OUTPUTS, 0)));
    C_TRY(alloc(s, &s->dout, act_floats(s, LBM_SURROGATE_OUTPUTS, 0)));
    // a[k+1] = output of conv k (k < 9) at level k/2 (conv8: level 4); decoder a[10+m] at level 3-m
    for (int k = 0; k < 9; ++k)
    {
        const int level = k < 8 ? k / 2 : 4;
        C_TRY(alloc(s, &s->a[k + 1], act_floats(s, kCout[k], level)));
        C_TRY(alloc(s, &s->da[k + 1], act_floats(s, kCout[k], level)));
    }
    for (int m = 0; m < 4; ++m)
    {
        C_TRY(alloc(s, &s->a[10 + m], act_floats(s, kCout[9 + m], 3 - m)));
        C_TRY(alloc(s, &s->da[10 + m], act_floats(s, kCout[9 + m], 3 - m)));
    }
    for (int l = 1; l <= 4; ++l)
        C_TRY(alloc(s, &s->p[l], act_floats(s, kCout[2 * l - 1], l)));
    size_t tmp = 0;
    for (int l = 1; l <= 4; ++l)
        tmp = std::max(tmp, act_floats(s, kCin[l == 4 ? 8 : 2 * l], l));
    C_TRY(alloc(s, &s->dtmp, tmp));
    C_TRY([&]() -> int {
        S_TRY(hipStreamSynchronize(s->stream));
        return LBM_OK;
    }());
#undef C_TRY
    *out = s;
    return LBM_OK;
}

int lbm_surrogate_init_params(lbm_surrogate *s, uint64_t seed)
{
    if (!s)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_init_params: null handle");
    std::vector<float> host(s->nparams, 0.f);
    uint64_t st = seed;
    for (int k = 0; k < kConvs; ++k)
    {
        const double stdev = std::sqrt(2.0 / (9.0 * kCin[k]));
        const size_t n = size_t(kCout[k]) * kCin[k] * 9;
        for (size_t i = 0; i < n; i += 2)
        {
            // Box-Muller pair
            const double u1 = std::max(uniform01(st), 1e-300), u2 = uniform01(st);
            const double r = std::sqrt(-2.0 * std::log(u1)), t = 2.0 * kPi * u2;
            host[s->w_off[k] + i] = float(stdev * r * std::cos(t));
            if (i + 1 < n)
                host[s->w_off[k] + i + 1] = float(stdev * r * std::sin(t));
        }
    }
    return lbm_surrogate_set_params(s, host.data(), host.size());
}

int lbm_surrogate_set_params(lbm_surrogate *s, const float *params, size_t count)
{
    if (!s || !params || count != s->nparams)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_set_params: count must equal the parameter count");
    S_TRY(hipMemcpyAsync(s->params, params, count * sizeof(float), hipMemcpyHostToDevice, s->stream));
    if (int rc = reset_adam(s))
        return rc;
    if (int rc = pack_all(s))
        return rc;
    S_TRY(hipStreamSynchronize(s->stream));
    return LBM_OK;
}

int lbm_surrogate_get_params(lbm_surrogate *s, float *params, size_t count)
{
    if (int rc = check_ready(s, "lbm_surrogate_get_params"))
        return rc;
    if (!params || count != s->nparams)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_get_params: count must equal the parameter count");
    S_TRY(hipMemcpyAsync(params, s->params, count * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    S_TRY(hipStreamSynchronize(s->stream));
    return LBM_OK;
}

static int predict(lbm_surrogate *s, const float *inputs, uint32_t batch, float *outputs, bool bf16)
{
    if (int rc = check_ready(s, "lbm_surrogate_predict"))
        return rc;
    if (!inputs || !outputs)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_predict: null buffer");
    const size_t hw = size_t(s->H) * s->W;
    S_TRY(hipEventRecord(s->ev0, s->stream));
    for (uint32_t b0 = 0; b0 < batch; b0 += uint32_t(s->Bmax))
    {
        const int B = int(std::min<uint32_t>(uint32_t(s->Bmax), batch - b0));
        S_TRY(hipMemcpyAsync(s->in, inputs + size_t(b0) * LBM_SURROGATE_INPUTS * hw,
                             size_t(B) * LBM_SURROGATE_INPUTS * hw * sizeof(float), hipMemcpyHostToDevice, s->stream));
        forward(s, B, bf16);
        S_TRY(hipGetLastError());
        const lbm_dev::HostPiece piece{outputs + size_t(b0) * LBM_SURROGATE_OUTPUTS * hw, s->out,
                                       size_t(B) * LBM_SURROGATE_OUTPUTS * hw * sizeof(float)};
        S_TRY(lbm_dev::download(&piece, 1, s->stream));
    }
    S_TRY(hipEventRecord(s->ev1, s->stream));
    S_TRY(hipStreamSynchronize(s->stream));
    float ms = 0.f;
    S_TRY(hipEventElapsedTime(&ms, s->ev0, s->ev1));
    s->last_ms = ms;
    return LBM_OK;
}

int lbm_surrogate_predict(lbm_surrogate *s, const float *inputs, uint32_t batch, float *outputs)
{
    return predict(s, inputs, batch, outputs, false);
}

int lbm_surrogate_predict_bf16(lbm_surrogate *s, const float *inputs, uint32_t batch, float *outputs)
{
    return predict(s, inputs, batch, outputs, true);
}

static int host_batch(lbm_surrogate *s, const float *inputs, const float *targets, uint32_t batch, double *norm,
                      const char *what)
{
    if (int rc = check_ready(s, what))
        return rc;
    if (!inputs || !targets || batch == 0 || batch > uint32_t(s->Bmax))
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, std::string(what) + ": batch must be in 1..max_batch");
    const size_t hw = size_t(s->H) * s->W;
    S_TRY(hipMemcpyAsync(s->in, inputs, size_t(batch) * LBM_SURROGATE_INPUTS * hw * sizeof(float),
                         hipMemcpyHostToDevice, s->stream));
    const unsigned blocks = std::min<unsigned>(kLossBlocks, elem_grid(size_t(batch) * hw));
    hipLaunchKernelGGL(k_mask_sum, dim3(blocks), dim3(256), 0, s->stream, s->in, s->loss_part, int(batch), int(hw));
    hipLaunchKernelGGL(k_loss_final, dim3(1), dim3(256), 0, s->stream, s->loss_part, int(blocks), 1.0,
                       s->loss_dev + 1, nullptr, 0);
    S_TRY(hipGetLastError());
    S_TRY(hipMemcpyAsync(s->tgt, targets, size_t(batch) * LBM_SURROGATE_OUTPUTS * hw * sizeof(float),
                         hipMemcpyHostToDevice, s->stream));
    double m = 0.0;
    S_TRY(hipMemcpyAsync(&m, s->loss_dev + 1, sizeof(double), hipMemcpyDeviceToHost, s->stream));
    S_TRY(hipStreamSynchronize(s->stream));
    if (!(m > 0.0))
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, std::string(what) + ": the batch has no fluid node");
    *norm = 1.0 / (double(LBM_SURROGATE_OUTPUTS) * m);
    return LBM_OK;
}

int lbm_surrogate_loss_grad(lbm_surrogate *s, const float *inputs, const float *targets, uint32_t batch,
                            double *loss, float *grad, size_t count)
{
    double norm = 0.0;
    if (int rc = host_batch(s, inputs, targets, batch, &norm, "lbm_surrogate_loss_grad"))
        return rc;
    if (!loss || !grad || count != s->nparams)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_loss_grad: bad output buffers");
    forward(s, int(batch));
    loss_backward(s, int(batch), norm, nullptr, 0);
    S_TRY(hipGetLastError());
    const lbm_dev::HostPiece pieces[2] = {{loss, s->loss_dev, sizeof(double)}, {grad, s->grad, count * sizeof(float)}};
    S_TRY(lbm_dev::download(pieces, 2, s->stream));
    return LBM_OK;
}

int lbm_surrogate_train_step(lbm_surrogate *s, const float *inputs, const float *targets, uint32_t batch,
                             float learning_rate, double *loss)
{
    double norm = 0.0;
    if (int rc = host_batch(s, inputs, targets, batch, &norm, "lbm_surrogate_train_step"))
        return rc;
    forward(s, int(batch));
    loss_backward(s, int(batch), norm, nullptr, 0);
    S_TRY(hipGetLastError());
    if (int rc = adam_step(s, learning_rate))
        return rc;
    if (loss)
        S_TRY(hipMemcpyAsync(loss, s->loss_dev, sizeof(double), hipMemcpyDeviceToHost, s->stream));
    S_TRY(hipStreamSynchronize(s->stream));
    return LBM_OK;
}

int lbm_surrogate_dataset_reserve(lbm_surrogate *s, size_t capacity)
{
    if (!s || capacity == 0)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_dataset_reserve: bad argument");
    const size_t hw = size_t(s->H) * s->W;
    (void)hipFree(s->ds_in);
    (void)hipFree(s->ds_tgt);
    s->ds_in = s->ds_tgt = nullptr;
    s->ds_cap = s->ds_n = 0;
    s->ds_fluid.clear();
    s->shuffle_seeded = false;
    S_TRY(hipMalloc(&s->ds_in, capacity * LBM_SURROGATE_INPUTS * hw * sizeof(float)));
    S_TRY(hipMalloc(&s->ds_tgt, capacity * LBM_SURROGATE_OUTPUTS * hw * sizeof(float)));
    s->ds_cap = capacity;
    return LBM_OK;
}

int lbm_surrogate_dataset_add(lbm_surrogate *s, const float *inputs, const float *targets, uint32_t count)
{
    if (!s || !inputs || !targets)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_dataset_add: bad argument");
    if (s->ds_n + count > s->ds_cap)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_dataset_add: capacity exceeded");
    const size_t hw = size_t(s->H) * s->W;
    for (uint32_t i = 0; i < count; ++i)
        s->ds_fluid.push_back(fluid_sum(inputs + size_t(i) * LBM_SURROGATE_INPUTS * hw, 1, hw));
    S_TRY(hipMemcpyAsync(s->ds_in + s->ds_n * LBM_SURROGATE_INPUTS * hw, inputs,
                         size_t(count) * LBM_SURROGATE_INPUTS * hw * sizeof(float), hipMemcpyHostToDevice, s->stream));
    S_TRY(hipMemcpyAsync(s->ds_tgt + s->ds_n * LBM_SURROGATE_OUTPUTS * hw, targets,
                         size_t(count) * LBM_SURROGATE_OUTPUTS * hw * sizeof(float), hipMemcpyHostToDevice,
                         s->stream));
    S_TRY(hipStreamSynchronize(s->stream));
    s->ds_n += count;
    s->shuffle_seeded = false;
    return LBM_OK;
}

size_t lbm_surrogate_dataset_size(const lbm_surrogate *s) { return s ? s->ds_n : 0; }

int lbm_surrogate_train(lbm_surrogate *s, uint32_t steps, uint32_t schedule_steps, uint32_t batch, float lr_max,
                        float lr_min, uint64_t seed, float *loss_history)
{
    if (int rc = check_ready(s, "lbm_surrogate_train"))
        return rc;
    if (batch == 0 || batch > uint32_t(s->Bmax) || s->ds_n < batch || schedule_steps == 0)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT,
                             "lbm_surrogate_train: batch must be in 1..max_batch and at most the dataset size, "
                             "schedule_steps > 0");
    if (steps == 0)
        return LBM_OK;
    if (s->history_cap < steps)
    {
        (void)hipFree(s->history);
        s->history = nullptr;
        s->history_cap = 0;
        S_TRY(hipMalloc(&s->history, size_t(steps) * sizeof(float)));
        s->history_cap = steps;
    }
    const size_t hw = size_t(s->H) * s->W;
    if (!s->shuffle_seeded)
    {
        s->perm.resize(s->ds_n);
        for (size_t i = 0; i < s->perm.size(); ++i)
            s->perm[i] = uint32_t(i);
        s->shuffle_state = seed;
        s->cursor = s->perm.size();
        s->shuffle_seeded = true;
    }
    std::vector<uint32_t> &perm = s->perm;
    const uint32_t warm = std::max<uint32_t>(1, std::min<uint32_t>(200, schedule_steps / 10));
    S_TRY(hipEventRecord(s->ev0, s->stream));
    for (uint32_t step = 0; step < steps; ++step)
    {
        if (s->cursor + batch > perm.size())
        {
            for (size_t i = perm.size() - 1; i > 0; --i)
                std::swap(perm[i], perm[splitmix64(s->shuffle_state) % (i + 1)]);
            s->cursor = 0;
        }
        const size_t cursor = s->cursor;
        double m = 0.0;
        for (uint32_t i = 0; i < batch; ++i)
        {
            const size_t id = perm[cursor + i];
            m += s->ds_fluid[id];
            S_TRY(hipMemcpyAsync(s->in + size_t(i) * LBM_SURROGATE_INPUTS * hw,
                                 s->ds_in + id * LBM_SURROGATE_INPUTS * hw, LBM_SURROGATE_INPUTS * hw * sizeof(float),
                                 hipMemcpyDeviceToDevice, s->stream));
            S_TRY(hipMemcpyAsync(s->tgt + size_t(i) * LBM_SURROGATE_OUTPUTS * hw,
                                 s->ds_tgt + id * LBM_SURROGATE_OUTPUTS * hw,
                                 LBM_SURROGATE_OUTPUTS * hw * sizeof(float), hipMemcpyDeviceToDevice, s->stream));
        }
        s->cursor += batch;
        if (!(m > 0.0))
            return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_train: a minibatch has no fluid node");
        const uint32_t g = s->sched_step++;
        double lr;
        if (g < warm)
            lr = lr_max * double(g + 1) / warm;
        else
        {
            const double t = std::min(1.0, double(g - warm) / std::max<uint32_t>(1, schedule_steps - warm));
            lr = lr_min + 0.5 * (lr_max - lr_min) * (1.0 + std::cos(kPi * t));
        }
        forward(s, int(batch));
        loss_backward(s, int(batch), 1.0 / (double(LBM_SURROGATE_OUTPUTS) * m), s->history, int(step));
        S_TRY(hipGetLastError());
        if (int rc = adam_step(s, float(lr)))
            return rc;
    }
    S_TRY(hipEventRecord(s->ev1, s->stream));
    if (loss_history)
        S_TRY(hipMemcpyAsync(loss_history, s->history, size_t(steps) * sizeof(float), hipMemcpyDeviceToHost,
                             s->stream));
    S_TRY(hipStreamSynchronize(s->stream));
    float ms = 0.f;
    S_TRY(hipEventElapsedTime(&ms, s->ev0, s->ev1));
    s->last_ms = ms;
    return LBM_OK;
}

int lbm_surrogate_last_ms(const lbm_surrogate *s, double *ms)
{
    if (!s || !ms)
        return lbm_set_error(LBM_ERR_INVALID_ARGUMENT, "lbm_surrogate_last_ms: bad argument");
    *ms = s->last_ms;
    return LBM_OK;
}

}  // extern "C"
