// 3x3 convolutions with 32 input and 32 output channels for the warm-start
// network: forward, backward-data and backward-weights on the gfx950 matrix
// cores (v_mfma_f32_16x16x32_bf16: BF16 operands, FP32 accumulation).
//
// Activations are NHWC in HBM (32 channels per pixel, zero padded when a
// layer has fewer), float32 or BF16; weights are prepared as BF16 in the
// layout [tap][out channel][in channel] (tap = 3*dy + dx).
//
// MFMA operand layout of the 16x16x32 BF16 instruction (lane l of 64):
//   A (16 x 32): row l%16, k = 8*(l/16) .. 8*(l/16)+7
//   B (32 x 16): col l%16, k = 8*(l/16) .. 8*(l/16)+7
//   D (16 x 16): col l%16, rows 4*(l/16) .. 4*(l/16)+3
#include "opy_common.h"

#include <algorithm>
#include <type_traits>

namespace opy {
namespace {

constexpr int kCh = 32;              // channels
constexpr int kTW = 32;              // output tile width of the forward kernels
constexpr int kHW = kTW + 2;
constexpr int kPixStride = kCh + 8;  // bf16 elements per LDS pixel (padding against bank conflicts)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// 16-byte accesses to FP32 arrays that are only known to be element aligned
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ inline __bf16 to_bf16(float v) { return (__bf16)v; }

// The warm start's first and last layers read and write the solver's packed
// buffers directly (image n of a group at n * stride elements):
//   first (kFirst): input channel 0 = f - 0.5, channel 1 = loglam[n], the
//   other 30 zero, i.e. the network's input encoding, formed while staging;
//   last (kLast): x = ((f - 0.5) + 0.5) + o0 and y = (o1, o2) per pixel, the
//   decoding of the output, with only the first 16 output channels computed.
enum { kPlain = 0, kFirst = 1, kLast = 2 };
struct ConvIO {
  const float* f;       // packed images
  int64_t stride;       // elements between consecutive images of the group
  const float* loglam;  // kFirst: per image
  float* xo;            // kLast: image n at xo + n * stride
  float* yo;            // kLast: image n at yo + 2 n * stride (pairs)
};

// ---- forward / backward-data -------------------------------------------------
// y[n,h,w,co] = act(b[co] + sum_{tap,ci} W[tap][co][ci] * x[n, h+dy-1, w+dx-1, ci])
// act: 0 none, 1 ReLU.  bias may be NULL.  kMask: y is zeroed where mask (of
// y's shape) is not positive, the ReLU backward of the layer below.  TX / TY:
// element type of x / y in HBM (float, or __bf16 for activations between
// layers: the operands are rounded to BF16 for the matrix cores anyway, so a
// BF16 copy of a layer's output gives the next layer the same operands at
// half the traffic).
//
// An implicit GEMM per tap, D (16 out channels x 16 pixels of a row) += W (16 x
// 32) * x (32 x 16).  A block of four wavefronts computes 32 x kTH output pixels;
// its input with the one-pixel halo sits in LDS as BF16, and the next tile's
// input is on its way into registers meanwhile.  What the layers move bounds
// them (64-128 B per pixel against 18.4 kflop), so everything else is kept off
// the path:
// - The weights of all taps stay in registers (72 of them), and an input row's
//   three column shifts are read from LDS once for the three output rows that
//   use them: with 16 rows 36 LDS reads per 144 matrix instructions of a
//   wavefront's tile.  With the weights in LDS and a read per tap they were 54
//   for 72, and LDS was busier than the matrix cores.
// - The rows of W are permuted so that lane (pixel l%16, l/16) ends up with the
//   8 consecutive output channels 8*(l/16)..: the results leave straight from
//   registers, 16 or 32 bytes per lane and whole pixels per quarter wavefront,
//   where they used to be staged through LDS between two barriers.
// - Consecutive tiles go to the blocks of one XCD, whose L2 then serves the
//   halos.
// 8 x 1024^2, BF16 in and out: 295 -> 203 us a layer (5.3 TB/s); 32 x 128^2,
// FP32: 44 -> 25 us (5.3 TB/s).
// Accumulation per output runs over dy, dx and the 32 input channels in this
// order in every instantiation, so all of them give the same bits.
template <int MODE, typename TX, typename TY, bool kMask, int kTH>
__global__ void __launch_bounds__(256, 2) conv3x3_kernel(const TX* __restrict__ x, TY* __restrict__ y,
                                                         const __bf16* __restrict__ wt,
                                                         const float* __restrict__ bias,
                                                         const float* __restrict__ mask, int N, int H, int W, int act,
                                                         ConvIO io) {
  constexpr int NJ = MODE == kLast ? 1 : 2;  // blocks of 16 output channels
  constexpr int RW = kTH / 4;                // output rows of a wavefront
  constexpr int NHP = kHW * (kTH + 2);       // pixels of a halo tile
  constexpr int NV = MODE == kFirst ? NHP : NHP * (kCh / 8);  // staged vectors (kFirst: image values)
  constexpr int NPF = (NV + 255) / 256;
  __shared__ __align__(16) __bf16 xs[MODE == kFirst ? 2 * NHP : NHP * kPixStride];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int tx = (W + kTW - 1) / kTW, ty = (H + kTH - 1) / kTH;
  const int ntiles = N * tx * ty;
  const int G = gridDim.x;
  const int first = (G % 8 == 0) ? ((int)blockIdx.x % 8) * (G / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;

  bf16x8 wr[9][NJ];  // row l%16 of block j is output channel 8*(l%16/4) + 4*j + l%4
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const __bf16* p = wt + (tap * kCh + 8 * (li >> 2) + 4 * j + (li & 3)) * kCh + 8 * lk;
      if ((reinterpret_cast<uintptr_t>(wt) & 15) == 0) {
        wr[tap][j] = *reinterpret_cast<const bf16x8*>(p);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) wr[tap][j][e] = p[e];
      }
    }
  float bv[4 * NJ];
#pragma unroll
  for (int e = 0; e < 4 * NJ; ++e) bv[e] = bias ? bias[8 * lk + e] : 0.f;

  auto origin = [&](int t, int& n, int& h0, int& w0) {
    n = t / (tx * ty);
    const int rem = t - n * tx * ty;
    h0 = (rem / tx) * kTH;
    w0 = (rem % tx) * kTW;
  };
  // the next tile's input: image values, BF16 vectors, or FP32 vectors (rounded on the way to LDS)
  float pf[MODE == kFirst ? NPF : 1];
  bf16x8 pv[MODE != kFirst && sizeof(TX) == 2 ? NPF : 1];
  f32x4 pa[MODE != kFirst && sizeof(TX) == 4 ? NPF : 1], pb[MODE != kFirst && sizeof(TX) == 4 ? NPF : 1];
  auto prefetch = [&](int t) {
    int n, h0, w0;
    origin(t, n, h0, w0);
#pragma unroll
    for (int i = 0; i < NPF; ++i) {
      const int e = tid + 256 * i;
      const int p = MODE == kFirst ? e : e >> 2;
      const int hh = h0 - 1 + p / kHW, ww = w0 - 1 + p % kHW;
      const bool in = p < NHP && hh >= 0 && hh < H && ww >= 0 && ww < W;
      if constexpr (MODE == kFirst) {
        pf[i] = in ? io.f[(int64_t)n * io.stride + (int64_t)hh * W + ww] : 0.f;
      } else {
        const TX* s = x + (((int64_t)n * H + hh) * W + ww) * kCh + 8 * (e & 3);
        if constexpr (sizeof(TX) == 2) {
          pv[i] = bf16x8{};
          if (in) pv[i] = *reinterpret_cast<const bf16x8*>(s);
        } else {
          f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
          if (in) {
            a = *reinterpret_cast<const f32x4*>(s);
            b = *reinterpret_cast<const f32x4*>(s + 4);
          }
          pa[i] = a;
          pb[i] = b;
        }
      }
    }
  };
  auto to_lds = [&](int t) {
    if constexpr (MODE == kFirst) {
      int n, h0, w0;
      origin(t, n, h0, w0);
      const __bf16 ll = to_bf16(io.loglam[n]);
#pragma unroll
      for (int i = 0; i < NPF; ++i) {
        const int p = tid + 256 * i;
        if (p >= NHP) continue;
        const int hh = h0 - 1 + p / kHW, ww = w0 - 1 + p % kHW;
        const bool in = hh >= 0 && hh < H && ww >= 0 && ww < W;
        xs[2 * p] = in ? to_bf16(pf[i] - 0.5f) : to_bf16(0.f);
        xs[2 * p + 1] = in ? ll : to_bf16(0.f);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NPF; ++i) {
        const int e = tid + 256 * i;
        if (e >= NV) continue;
        bf16x8 v;
        if constexpr (sizeof(TX) == 2) v = pv[i];
        else v = __builtin_convertvector(__builtin_shufflevector(pa[i], pb[i], 0, 1, 2, 3, 4, 5, 6, 7), bf16x8);
        *reinterpret_cast<bf16x8*>(xs + (e >> 2) * kPixStride + 8 * (e & 3)) = v;
      }
    }
  };

  if (first < ntiles) prefetch(first);
  for (int t = first; t < ntiles; t += G) {
    __syncthreads();  // every wavefront is done with the previous tile
    to_lds(t);
    __syncthreads();
    int n, h0, w0;
    origin(t, n, h0, w0);
    float fc[MODE == kLast ? 2 * RW : 1];
    if constexpr (MODE == kLast) {
      // the pixels' own image values, on their way before the next tile's input
#pragma unroll
      for (int k = 0; k < 2 * RW; ++k) {
        const int h = h0 + wave * RW + k % RW, w = w0 + (k / RW) * 16 + li;
        fc[k] = (lk == 0 && h < H && w < W) ? io.f[(int64_t)n * io.stride + (int64_t)h * W + w] : 0.f;
      }
    }
    if (t + G < ntiles) prefetch(t + G);
#pragma unroll
    for (int cb = 0; cb < kTW / 16; ++cb) {
      // wavefront `wave` has the output rows RW*wave .. RW*wave + RW-1 of the tile
      f32x4 acc[RW][NJ];
#pragma unroll
      for (int m = 0; m < RW; ++m)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < RW + 2; ++i)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const int p = (wave * RW + i) * kHW + cb * 16 + li + dx;
          bf16x8 b;
          if constexpr (MODE == kFirst) {
            u32x4 v = {0u, 0u, 0u, 0u};
            const uint32_t q = *reinterpret_cast<const uint32_t*>(xs + 2 * p);
            v[0] = lk == 0 ? q : 0u;
            b = __builtin_bit_cast(bf16x8, v);
          } else {
            b = *reinterpret_cast<const bf16x8*>(xs + p * kPixStride + 8 * lk);
          }
#pragma unroll
          for (int m = 0; m < RW; ++m) {
            const int dy = i - m;
            if (dy < 0 || dy > 2) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[3 * dy + dx][j], b, acc[m][j], 0, 0, 0);
          }
        }
      const int w = w0 + cb * 16 + li;
#pragma unroll
      for (int m = 0; m < RW; ++m) {
        const int h = h0 + wave * RW + m;
        if (h >= H || w >= W) continue;
        float v[4 * NJ];
#pragma unroll
        for (int e = 0; e < 4 * NJ; ++e) {
          v[e] = acc[m][e >> 2][e & 3] + bv[e];
          if (act == 1) v[e] = v[e] > 0.f ? v[e] : 0.f;
        }
        if constexpr (MODE == kLast) {
          if (lk == 0) {
            const int64_t q = (int64_t)n * io.stride + (int64_t)h * W + w;
            io.xo[q] = ((fc[cb * RW + m] - 0.5f) + 0.5f) + v[0];
            *reinterpret_cast<float2*>(io.yo + 2 * q) = make_float2(v[1], v[2]);
          }
        } else {
          const int64_t o = (((int64_t)n * H + h) * W + w) * kCh + 8 * lk;
          if constexpr (kMask) {
            const f32x4 m0 = *reinterpret_cast<const f32x4u*>(mask + o);
            const f32x4 m1 = *reinterpret_cast<const f32x4u*>(mask + o + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (!((e < 4 ? m0[e & 3] : m1[e & 3]) > 0.f)) v[e] = 0.f;
          }
          if constexpr (sizeof(TY) == 2) {
            bf16x8 q;
#pragma unroll
            for (int e = 0; e < 8; ++e) q[e] = to_bf16(v[e]);
            *reinterpret_cast<bf16x8*>(y + o) = q;
          } else {
            *reinterpret_cast<f32x4u*>(y + o) = f32x4{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<f32x4u*>(y + o + 4) = f32x4{v[4], v[5], v[6], v[7]};
          }
        }
      }
    }
  }
}

// Two blocks per CU hold the weights and the next tile's input in registers; each block walks
// several tiles. Output rows per tile, measured on a 32 x 128^2 batch (FP32 in and out) and on
// 8 x 1024^2 (BF16): FP32 input 8 rows 25 us a layer (5.3 TB/s), 16 rows 28 us (the next tile takes
// 80 registers), without loading ahead 28-30 us; BF16 input 16 rows 203 us a layer (5.3 TB/s),
// 8 rows 212 us, without loading ahead 245 us.
template <int MODE, typename TX, typename TY, bool kMask>
void launch_conv(const TX* x, TY* y, const void* wt, const float* bias, const float* mask, int N, int H, int W,
                 int act, const ConvIO& io, int grid, hipStream_t st) {
  constexpr int TH = sizeof(TX) == 4 ? 8 : 16;
  constexpr int kMost = 512;
  const int64_t tiles = (int64_t)N * ((H + TH - 1) / TH) * ((W + kTW - 1) / kTW);
  int64_t g = std::min<int64_t>(std::min(grid, kMost), tiles);
  if (g > 8) g -= g % 8;  // whole rounds of the 8 XCDs
  hipLaunchKernelGGL((conv3x3_kernel<MODE, TX, TY, kMask, TH>), dim3((unsigned)g), dim3(256), 0, st, x, y,
                     static_cast<const __bf16*>(wt), bias, mask, N, H, W, act, io);
}

// ---- backward-weights ----------------------------------------------------------
// dW[tap][co][ci] = sum_{n,h,w} g[n,h,w,co] * x[n, h+dy-1, w+dx-1, ci]   (partials per block)
// dbias[co] = sum g[..., co]  (partials per block, slot 9*32*32 + co)
// As a GEMM per tap: D (co x ci) += A (co x pixels) * B (pixels x ci), 32 pixels
// of a row per matrix instruction.  A block walks tiles of 32 x 8 pixels, staged
// in LDS channel-major as BF16 (a thread takes 4 channels of 8 consecutive
// pixels from NHWC memory and writes one 16-byte vector per channel); wavefront
// (i, j) owns the 16 x 16 block (i, j) of every tap's matrix.  The operands of
// the three column shifts come from one aligned 16-byte and one 4-byte LDS read
// by byte alignment, and an input row serves the three output rows it borders,
// so a row costs 3 LDS reads for 9 matrix instructions.  32 x 128^2: 107 -> 35 us
// a layer, 4.3 TB/s of x, g and the partials; the matrix cores are busy for 13% of
// it, the LDS for 40% (70% of that bank conflicts).
constexpr int kGW = 32, kGH = 8;          // tile
constexpr int kGP = 40;                   // bf16 elements per (row, channel) in LDS, 34 / 32 used
__global__ void __launch_bounds__(256) conv3x3_wgrad_kernel(const float* __restrict__ x, const float* __restrict__ g,
                                                            float* __restrict__ partials, int N, int H, int W) {
  __shared__ __align__(16) __bf16 xs[(kGH + 2) * kCh * kGP];
  __shared__ __align__(16) __bf16 gs[kGH * kCh * kGP];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int ib = wave >> 1, jb = wave & 1;  // this wavefront's co and ci block
  const int tx = (W + kGW - 1) / kGW, ty = (H + kGH - 1) / kGH;
  const int ntiles = N * tx * ty;
  const int G = gridDim.x;
  const int first = (G % 8 == 0) ? ((int)blockIdx.x % 8) * (G / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;
  f32x4 acc[9];
#pragma unroll
  for (int a = 0; a < 9; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 bacc = {0.f, 0.f, 0.f, 0.f};  // FP32 bias-gradient partial of the 4 channels this thread stages
  // 4 channels (quad c4) of the 8 pixels w .. w+7 of row h, of which those inside the image and below nw
  auto load8 = [&](const float* base, int n, int h, int w, int c4, int nw, f32x4 (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (e < nw && h >= 0 && h < H && w + e >= 0 && w + e < W)
        v[e] = *reinterpret_cast<const f32x4u*>(base + (((int64_t)n * H + h) * W + w + e) * kCh + 4 * c4);
    }
  };
  auto put8 = [&](__bf16* d, const f32x4 (&v)[8]) {  // d: (row, channel 4*c4, pixel group)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      bf16x8 q;
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = to_bf16(v[e][k]);
      *reinterpret_cast<bf16x8*>(d + k * kGP) = q;
    }
  };
  for (int t = first; t < ntiles; t += G) {
    const int n = t / (tx * ty);
    const int rem = t - n * tx * ty;
    const int h0 = (rem / tx) * kGH, w0 = (rem % tx) * kGW;
    constexpr int NX = (kGH + 2) * 5 * (kCh / 4);  // pieces of the x tile (5 pixel groups per row)
    static_assert(kGH * (kGW / 8) * (kCh / 4) == 256 && NX > 256 && NX <= 512, "one g piece and up to two of x a thread");
    const int c4 = tid & 7, gq = (tid >> 3) & 3, gr = tid >> 5;
    const int e0 = tid >> 3, e1 = (tid + 256) >> 3;
    f32x4 vg[8], va[8], vb[8];
    load8(g, n, h0 + gr, w0 + 8 * gq, c4, 8, vg);
    load8(x, n, h0 - 1 + e0 / 5, w0 - 1 + 8 * (e0 % 5), c4, e0 % 5 == 4 ? 2 : 8, va);
    const bool two = tid + 256 < NX;
    load8(x, n, two ? h0 - 1 + e1 / 5 : -1, w0 - 1 + 8 * (e1 % 5), c4, e1 % 5 == 4 ? 2 : 8, vb);
    __syncthreads();  // every wavefront is done with the previous tile
    put8(gs + (gr * kCh + 4 * c4) * kGP + 8 * gq, vg);
    put8(xs + ((e0 / 5) * kCh + 4 * c4) * kGP + 8 * (e0 % 5), va);
    if (two) put8(xs + ((e1 / 5) * kCh + 4 * c4) * kGP + 8 * (e1 % 5), vb);
#pragma unroll
    for (int e = 0; e < 8; ++e) bacc += vg[e];
    __syncthreads();
    bf16x8 ga[kGH];  // g rows of this wavefront's co block
#pragma unroll
    for (int i = 0; i < kGH + 2; ++i) {
      if (i < kGH) ga[i] = *reinterpret_cast<const bf16x8*>(gs + (i * kCh + ib * 16 + li) * kGP + 8 * lk);
      const __bf16* s = xs + (i * kCh + jb * 16 + li) * kGP + 8 * lk;
      const u32x4 d = *reinterpret_cast<const u32x4*>(s);
      const uint32_t d4 = *reinterpret_cast<const uint32_t*>(s + 8);
      u32x4 b[3];
      b[0] = d;
      b[1] = u32x4{__builtin_amdgcn_alignbyte(d[1], d[0], 2), __builtin_amdgcn_alignbyte(d[2], d[1], 2),
                   __builtin_amdgcn_alignbyte(d[3], d[2], 2), __builtin_amdgcn_alignbyte(d4, d[3], 2)};
      b[2] = u32x4{d[1], d[2], d[3], d4};
#pragma unroll
      for (int dy = 0; dy < 3; ++dy) {
        const int r = i - dy;
        if (r < 0 || r >= kGH) continue;
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
          acc[3 * dy + dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga[r], __builtin_bit_cast(bf16x8, b[dx]),
                                                                     acc[3 * dy + dx], 0, 0, 0);
      }
    }
  }
  // write this block's partials: D rows = co (4*(l/16)+r within the 16-block), cols = ci (l%16)
  float* pb = partials + (int64_t)blockIdx.x * (9 * kCh * kCh + kCh);
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int r = 0; r < 4; ++r) pb[(tap * kCh + ib * 16 + 4 * lk + r) * kCh + jb * 16 + li] = acc[tap][r];
  __syncthreads();
  f32x4* bs = reinterpret_cast<f32x4*>(xs);
  bs[tid] = bacc;
  __syncthreads();
  if (tid < kCh) {
    float sb = 0.f;
    for (int k = 0; k < 32; ++k) sb += bs[(tid >> 2) + 8 * k][tid & 3];
    pb[9 * kCh * kCh + tid] = sb;
  }
}

// Sum of nb partial vectors of length len in a fixed order: a block has 64
// columns and 16 segments of the partials, each summed in order and then folded
// through LDS, so that 1024 threads' loads are in flight per 64 columns (one
// thread per column walking all the partials took 475 us for 2048 of length
// 9248, with 9248 loads in flight on the chip).  kTrans: the partials are a
// layer's [tap][co][ci] and bias gradients, and out gets [tap][ci][co].
template <bool kTrans>
__global__ void __launch_bounds__(1024) sum_partials_kernel(const float* __restrict__ partials, int nb, int len,
                                                            float* __restrict__ out) {
  __shared__ float sm[16][64];
  const int col = threadIdx.x & 63, seg = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + col;
  const int per = (nb + 15) / 16;
  const int lo = min(nb, seg * per), hi = min(nb, lo + per);
  float s = 0.f;
  if (i < len) {
    const float* p = partials + i;
    int b = lo;
    for (; b + 8 <= hi; b += 8) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = p[(int64_t)(b + k) * len];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
    for (; b < hi; ++b) s += p[(int64_t)b * len];
  }
  sm[seg][col] = s;
  __syncthreads();
  if (seg != 0 || i >= len) return;
  s = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) s += sm[k][col];
  int o = i;
  if (kTrans && i < 9 * kCh * kCh) o = (i & ~(kCh * kCh - 1)) + (i % kCh) * kCh + (i / kCh) % kCh;
  out[o] = s;
}

// weights: master W[tap][ci][co] (float) -> bf16 [tap][co][ci] (transpose=0, forward)
// or the backward-data weights Wb[tap][ci][co] = W[8-tap][ci][co] in the [tap][out=ci][in=co] layout
__device__ inline __bf16 prep_weight(const float* __restrict__ w, int e, int flip) {
  const int tap = e / (kCh * kCh);
  const int r = e % (kCh * kCh);
  const int o = r / kCh, i = r % kCh;  // out[tap][o][i]
  return to_bf16(flip ? w[((8 - tap) * kCh + o) * kCh + i]   // W[8-tap][ci=o][co=i]
                      : w[(tap * kCh + i) * kCh + o]);       // W[tap][ci=i][co=o]
}
__global__ void prep_weights_kernel(const float* __restrict__ w, __bf16* __restrict__ out, int flip) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < 9 * kCh * kCh) out[e] = prep_weight(w, e, flip);
}
// every layer's forward and backward-data weights in one launch (blockIdx.y = layer)
__global__ void prep_all_kernel(const float* __restrict__ params, int64_t per, __bf16* __restrict__ wf,
                                __bf16* __restrict__ wb) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 9 * kCh * kCh) return;
  const float* w = params + blockIdx.y * per;
  wf[blockIdx.y * (int64_t)(9 * kCh * kCh) + e] = prep_weight(w, e, 0);
  wb[blockIdx.y * (int64_t)(9 * kCh * kCh) + e] = prep_weight(w, e, 1);
}

// g = g * (y > 0): ReLU backward through the stored activation
__global__ void relu_bwd_kernel(float* __restrict__ g, const float* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !(y[i] > 0.f)) g[i] = 0.f;
}

// Adam step on n parameters (FP32 master copy)
__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, int n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// weighted squared error over the first nc channels of NHWC-32 tensors:
// loss = sum_{p, c<nc} wc[c]*(out - tgt)^2 / npix, grad = d loss / d out (zero for c >= nc);
// per-block loss partials in FP64.  A thread takes 4 channels; only the first
// quad of a pixel is read, the other seven are written as zeros.
__global__ void __launch_bounds__(256) mse_kernel(const float* __restrict__ out, const float* __restrict__ tgt,
                                                  float* __restrict__ grad, int64_t npix, int nc, float w0, float w1,
                                                  float w2, double* __restrict__ partials) {
  __shared__ double sm[4];
  const int64_t n = npix * (kCh / 4);
  const float inv = 1.0f / (float)npix;
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    f32x4 gv = {0.f, 0.f, 0.f, 0.f};
    if (i % (kCh / 4) == 0) {
      const f32x4 a = *reinterpret_cast<const f32x4u*>(out + 4 * i), b = *reinterpret_cast<const f32x4u*>(tgt + 4 * i);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (c >= nc) continue;
        const float wc = c == 0 ? w0 : (c == 1 ? w1 : w2);
        const float d = a[c] - b[c];
        s += (double)wc * (double)d * (double)d;
        gv[c] = 2.f * wc * d * inv;
      }
    }
    *reinterpret_cast<f32x4u*>(grad + 4 * i) = gv;
  }
  s = block_sum(s, sm);
  if (threadIdx.x == 0) partials[blockIdx.x] = s / (double)npix;
}

}  // namespace
}  // namespace opy

using namespace opy;

OPY_API int opy_mse3_f32(const float* out, const float* tgt, float* grad, int64_t npix, int nc, double w0, double w1,
                         double w2, double* partials, int grid, void* s) {
  if (!out || !tgt || !grad || !partials || npix < 1 || nc < 1 || nc > 3 || grid < 1)
    return fail(kInvalid, "mse3: bad arguments");
  hipLaunchKernelGGL(mse_kernel, dim3(grid), dim3(256), 0, as_stream(s), out, tgt, grad, npix, nc, (float)w0,
                     (float)w1, (float)w2, partials);
  return check_launch("mse3");
}

OPY_API int opy_conv3x3_fwd_bf16(const float* x, float* y, const void* wt, const float* bias, int N, int H, int W,
                                 int act, int grid, void* s) {
  if (!x || !y || !wt || N < 1 || H < 1 || W < 1 || grid < 1) return fail(kInvalid, "conv3x3_fwd: bad arguments");
  if (x == y) return fail(kInvalid, "conv3x3_fwd: in-place convolution is not supported");
  if ((reinterpret_cast<uintptr_t>(x) & 15) != 0) return fail(kInvalid, "conv3x3_fwd: input must be 16-byte aligned");
  launch_conv<kPlain, float, float, false>(x, y, wt, bias, nullptr, N, H, W, act, ConvIO{}, grid, as_stream(s));
  return check_launch("conv3x3_fwd");
}
OPY_API int opy_conv3x3_bwd_data(const float* g, float* y, const void* wt, const float* mask, int N, int H, int W,
                                 int grid, void* s) {
  if (!g || !y || !wt || !mask || N < 1 || H < 1 || W < 1 || grid < 1)
    return fail(kInvalid, "conv3x3_bwd_data: bad arguments");
  if (g == y || mask == y) return fail(kInvalid, "conv3x3_bwd_data: the output must not alias an input");
  if ((reinterpret_cast<uintptr_t>(g) & 15) != 0)
    return fail(kInvalid, "conv3x3_bwd_data: input must be 16-byte aligned");
  launch_conv<kPlain, float, float, true>(g, y, wt, nullptr, mask, N, H, W, 0, ConvIO{}, grid, as_stream(s));
  return check_launch("conv3x3_bwd_data");
}
OPY_API int opy_conv3x3_fwd_io(const void* x, void* y, const void* wt, const float* bias, int N, int H, int W,
                               int act, int x_bf16, int y_bf16, int grid, void* s) {
  if (!x || !y || !wt || N < 1 || H < 1 || W < 1 || grid < 1) return fail(kInvalid, "conv3x3_fwd_io: bad arguments");
  if (x == y) return fail(kInvalid, "conv3x3_fwd_io: in-place convolution is not supported");
  if ((reinterpret_cast<uintptr_t>(x) & 15) != 0) return fail(kInvalid, "conv3x3_fwd_io: input must be 16-byte aligned");
  if (y_bf16 && (reinterpret_cast<uintptr_t>(y) & 15) != 0)
    return fail(kInvalid, "conv3x3_fwd_io: BF16 output must be 16-byte aligned");
  const __bf16* w = static_cast<const __bf16*>(wt);
  hipStream_t st = as_stream(s);
  const __bf16* xh = static_cast<const __bf16*>(x);
  const float* xf = static_cast<const float*>(x);
  __bf16* yh = static_cast<__bf16*>(y);
  float* yf = static_cast<float*>(y);
  if (x_bf16 && y_bf16)
    launch_conv<kPlain, __bf16, __bf16, false>(xh, yh, w, bias, nullptr, N, H, W, act, ConvIO{}, grid, st);
  else if (x_bf16)
    launch_conv<kPlain, __bf16, float, false>(xh, yf, w, bias, nullptr, N, H, W, act, ConvIO{}, grid, st);
  else if (y_bf16)
    launch_conv<kPlain, float, __bf16, false>(xf, yh, w, bias, nullptr, N, H, W, act, ConvIO{}, grid, st);
  else
    launch_conv<kPlain, float, float, false>(xf, yf, w, bias, nullptr, N, H, W, act, ConvIO{}, grid, st);
  return check_launch("conv3x3_fwd_io");
}

OPY_API int opy_conv3x3_first(const float* f, int64_t stride, const float* loglam, void* y, const void* wt,
                              const float* bias, int N, int H, int W, int grid, void* s) {
  if (!f || !loglam || !y || !wt || N < 1 || H < 1 || W < 1 || grid < 1 || stride < (int64_t)H * W)
    return fail(kInvalid, "conv3x3_first: bad arguments");
  if ((reinterpret_cast<uintptr_t>(y) & 15) != 0) return fail(kInvalid, "conv3x3_first: output must be 16-byte aligned");
  ConvIO io{f, stride, loglam, nullptr, nullptr};
  launch_conv<kFirst, __bf16, __bf16, false>(static_cast<const __bf16*>(nullptr), static_cast<__bf16*>(y), wt, bias, nullptr, N, H, W, 1, io, grid, as_stream(s));
  return check_launch("conv3x3_first");
}
OPY_API int opy_conv3x3_last(const void* x, const float* f, int64_t stride, float* xo, float* yo, const void* wt,
                             const float* bias, int N, int H, int W, int grid, void* s) {
  if (!x || !f || !xo || !yo || !wt || N < 1 || H < 1 || W < 1 || grid < 1 || stride < (int64_t)H * W)
    return fail(kInvalid, "conv3x3_last: bad arguments");
  if ((reinterpret_cast<uintptr_t>(x) & 15) != 0) return fail(kInvalid, "conv3x3_last: input must be 16-byte aligned");
  if ((reinterpret_cast<uintptr_t>(yo) & 7) != 0) return fail(kInvalid, "conv3x3_last: yo must be 8-byte aligned");
  ConvIO io{f, stride, nullptr, xo, yo};
  launch_conv<kLast, __bf16, __bf16, false>(static_cast<const __bf16*>(x), static_cast<__bf16*>(nullptr), wt, bias, nullptr, N, H, W, 0, io, grid, as_stream(s));
  return check_launch("conv3x3_last");
}

OPY_API int opy_conv3x3_wgrad_bf16(const float* x, const float* g, float* partials, int N, int H, int W, int grid,
                                   void* s) {
  if (!x || !g || !partials || N < 1 || H < 1 || W < 1 || grid < 1) return fail(kInvalid, "conv3x3_wgrad: bad arguments");
  hipLaunchKernelGGL(conv3x3_wgrad_kernel, dim3(grid), dim3(256), 0, as_stream(s), x, g, partials, N, H, W);
  return check_launch("conv3x3_wgrad");
}

OPY_API int opy_sum_partials_f32(const float* partials, int nb, int len, float* out, void* s) {
  if (!partials || !out || nb < 1 || len < 1) return fail(kInvalid, "sum_partials: bad arguments");
  hipLaunchKernelGGL(sum_partials_kernel<false>, dim3((len + 63) / 64), dim3(1024), 0, as_stream(s), partials, nb, len,
                     out);
  return check_launch("sum_partials");
}
OPY_API int opy_conv3x3_grad_reduce(const float* partials, int nb, float* out, void* s) {
  if (!partials || !out || nb < 1) return fail(kInvalid, "conv3x3_grad_reduce: bad arguments");
  constexpr int len = 9 * kCh * kCh + kCh;
  hipLaunchKernelGGL(sum_partials_kernel<true>, dim3((len + 63) / 64), dim3(1024), 0, as_stream(s), partials, nb, len,
                     out);
  return check_launch("conv3x3_grad_reduce");
}
OPY_API int opy_conv3x3_prep_all(const float* params, int64_t per, int layers, void* wf, void* wb, void* s) {
  if (!params || !wf || !wb || layers < 1 || per < 9 * kCh * kCh) return fail(kInvalid, "conv3x3_prep_all: bad arguments");
  hipLaunchKernelGGL(prep_all_kernel, dim3((9 * kCh * kCh + 255) / 256, layers), dim3(256), 0, as_stream(s), params, per,
                     static_cast<__bf16*>(wf), static_cast<__bf16*>(wb));
  return check_launch("conv3x3_prep_all");
}

OPY_API int opy_conv3x3_prep_weights(const float* w, void* out, int flip, void* s) {
  if (!w || !out) return fail(kInvalid, "prep_weights: null pointer");
  hipLaunchKernelGGL(prep_weights_kernel, dim3((9 * 32 * 32 + 255) / 256), dim3(256), 0, as_stream(s), w,
                     static_cast<__bf16*>(out), flip);
  return check_launch("prep_weights");
}

OPY_API int opy_relu_bwd_f32(float* g, const float* y, int64_t n, void* s) {
  if (n > 0 && (!g || !y)) return fail(kInvalid, "relu_bwd: null pointer");
  if (n > 0)
    hipLaunchKernelGGL(relu_bwd_kernel, dim3(grid_for(n)), dim3(256), 0, as_stream(s), g, y, n);
  return check_launch("relu_bwd");
}

OPY_API int opy_adam_f32(float* p, const float* g, float* m, float* v, int n, double lr, double b1, double b2,
                         double eps, int step, void* s) {
  if (n < 1 || !p || !g || !m || !v || step < 1) return fail(kInvalid, "adam: bad arguments");
  const float c1 = (float)(1.0 - pow(b1, step)), c2 = (float)(1.0 - pow(b2, step));
  hipLaunchKernelGGL(adam_kernel, dim3((n + 255) / 256), dim3(256), 0, as_stream(s), p, g, m, v, n, (float)lr,
                     (float)b1, (float)b2, (float)eps, c1, c2);
  return check_launch("adam");
}
