// shy_nn.hip -- BF16 MFMA kernels of the discharge/momentum surrogate (gfx950).
//
// Activations are NHWC bf16 (channels contiguous).  A 3x3 (pad 1) or 1x1
// convolution is an implicit GEMM: M = pixels, N = output channels,
// K = taps x input channels (tap-major), weights stored Wt[Cout][K] so both
// MFMA operands load 8 consecutive k as one 16-byte vector.  Every product
// runs on v_mfma_f32_16x16x32_bf16 with FP32 accumulation.  Lane layout of
// that instruction (checked on the device): lane l holds A[l%16][(l/16)*8+i],
// B[(l/16)*8+i][l%16] for i < 8 and C[(l/16)*4+i][l%16] for i < 4.
//
//   conv_tiles_kernel  3x3 forward / data gradient of every layer of 32-channel
//                      multiples, 16x16 pixel tiles (16x8 where all of those
//                      run at once): persistent blocks (three per CU, 32 output channels
//                      each) over the tiles, patch and weights staged in LDS,
//                      the next chunk's patch loaded into registers during
//                      the current chunk's MFMAs; decoder inputs read as
//                      [up2(x), skip] from two tensors; optionally a 1x1
//                      head on the rounded output, or its 2x2 average pool
//                      (pairs of rows in a lane, pairs of columns across
//                      lanes l and l ^ 1)
//   conv_pf_kernel     the same arithmetic with one tile per block, for 1x1
//                      convolutions and rows beyond the tile loop's offsets
//   conv_c8_kernel     the 8-channel first layer, four taps per MFMA k-step
//   conv_fwd_kernel    direct-load convolution of the remaining shapes (the
//                      head's data gradient)
//   epilogue           bias, an optional residual and ReLU, bf16 or f32
//                      store; for the data gradient (the forward kernels on
//                      weights flipped by flip_weights_kernel or written so
//                      by Adam) the residual gradient and the ReLU mask
//   wgrad_lds_kernel   dW[co][k] = sum_p g[p][co] x[p + tap][ci]: K = pixels,
//   conv_wgrad_kernel  staged through LDS (both operands need 8 consecutive
//                      pixels per lane: transposed LDS reads; the second loads
//                      directly), split over pixel ranges into FP32 partials
//                      that wgrad_reduce_kernel sums in a fixed order; both
//                      launches of the first take the bias gradient along
//   elementwise        ReLU backward, 2x2 average pool, nearest upsample,
//                      channel concat/split, the fused passes between two
//                      stages of the backward, bias gradient, MSE loss, Adam
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <string>

#include "../../include/shy_nn.h"

// Split-K partials of shy_nn_conv_wgrad_noalloc: SHY_NN_NOALLOC_FLOATS
// floats (16 MiB) on every device the library runs on, held until the
// process ends.  On the host this name is a stand-in, not a device address:
// host code uses only the address hipGetSymbolAddress returns for the
// current device (noalloc_scratch below).
static __device__ __align__(256) float scratch[SHY_NN_NOALLOC_FLOATS];

namespace shy_nn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
  return z;
}

__device__ inline bf16x8 load8(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

__device__ inline f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct ConvArgs {
  const __bf16* __restrict__ x;    // [P][Cin], P = N*H*W
  const __bf16* __restrict__ w;    // [Cout][K]
  const float* __restrict__ bias;  // [Cout] or null
  const __bf16* __restrict__ res;  // [P][Cout] or null (added before the ReLU)
  __bf16* y_bf;                    // [P][Cout] (one of y_bf / y_f)
  float* y_f;
  int N, H, W, Cin, Cout, K;
  int relu;
  // When x2 is set (UPCAT instantiations), the input is the concatenation of
  // a nearest x2 upsample of x ([N][H/2][W/2][C1]) and x2 ([N][H][W][Cin-C1]).
  const __bf16* __restrict__ x2;
  int C1;
  // Backward-pass epilogue of the LDS-staged kernels (bf16 output): after
  // rounding, gres ([P][Cout]) is added (in float, rounded again) and the
  // result is zeroed where mask ([P][Cout]) is not positive: the bits of
  // shy_nn_add then shy_nn_relu_bwd on the rounded output.
  const __bf16* __restrict__ gres;
  const __bf16* __restrict__ mask;
  // When head_w is set (HEAD instantiations, 32 output channels, BF16 output):
  // the epilogue also applies a 1x1 convolution to the rounded output,
  // head_y [P][head_c] (FP32) = head_b + head_w [head_c][32] . y, with one
  // MFMA per row of pixels; y_bf may then be null (y not stored).
  const __bf16* __restrict__ head_w = nullptr;
  const float* __restrict__ head_b = nullptr;
  float* head_y = nullptr;
  int head_c = 0;
  // When pool_y is set (conv_tiles_kernel, H and W even): also the 2x2
  // average of the rounded output, [N][H/2][W/2][Cout], with the bits of
  // pool2_fwd_v8_kernel on y.
  __bf16* pool_y = nullptr;
};

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// One lane's 4 consecutive output channels co..co+3 of output element o:
// bias, residual (before rounding), ReLU, then the store, FP32 or BF16 (with
// the backward-pass residual and mask after rounding).  Returns the BF16 values
// (zeros for an FP32 output); with HEAD a null y_bf stores nothing.
template <bool HEAD>
__device__ inline bf16x4 store_out4(const ConvArgs& a, size_t o, int co, const f32x4& acc) {
  float v[4];
  // the lane's 4 biases in one load: co is a multiple of 4 and the entry
  // points require a 16-byte aligned bias
  const float4 b = a.bias ? *reinterpret_cast<const float4*>(a.bias + co)
                          : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  v[0] = acc[0] + b.x;
  v[1] = acc[1] + b.y;
  v[2] = acc[2] + b.z;
  v[3] = acc[3] + b.w;
  if (a.res) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += (float)a.res[o + i];
  }
  if (a.relu) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
  }
  bf16x4 q = {};
  if (a.y_f) {
    *reinterpret_cast<float4*>(a.y_f + o) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = (__bf16)v[i];
    if (a.gres) {
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = (__bf16)((float)q[i] + (float)a.gres[o + i]);
    }
    if (a.mask) {
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = (float)a.mask[o + i] > 0.0f ? q[i] : (__bf16)0.0f;
    }
    if (!HEAD || a.y_bf) *reinterpret_cast<bf16x4*>(a.y_bf + o) = q;
  }
  return q;
}

// The 1x1 head on a tile's rounded 32-channel output q (ConvArgs::head_w),
// one MFMA per row of 16 pixels: the output channels are the M operand and
// the pixels the N operand, and the K operand takes each lane's own 8
// channels in the order it holds them, 4g..4g+3 then 16+4g..16+4g+3 for
// lane group g = lane/16, so the rounded output needs no exchange; the
// head's weights are read in that order.  Lane holds head channels
// 4(lane/16) + i of pixel lane%16.
template <int NT>
__device__ inline void conv_head(const ConvArgs& a, const bf16x4 (&q)[2][NT], int n, int y0,
                                 int x0, int wave, int lane) {
  const int hc = a.head_c, o = lane & 15, g = lane >> 4;
  // two 8-byte loads (head_w is 16-byte aligned, rows of 32)
  bf16x4 w0, w1;
#pragma unroll
  for (int j = 0; j < 4; ++j) w0[j] = w1[j] = (__bf16)0.0f;
  if (o < hc) {
    w0 = *reinterpret_cast<const bf16x4*>(a.head_w + o * 32 + 4 * g);
    w1 = *reinterpret_cast<const bf16x4*>(a.head_w + o * 32 + 16 + 4 * g);
  }
  bf16x8 A;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    A[j] = w0[j];
    A[4 + j] = w1[j];
  }
  const int gx = x0 + (lane & 15), oc = 4 * g;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    bf16x8 B;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      B[j] = q[0][t][j];
      B[4 + j] = q[1][t][j];
    }
    const f32x4 h = mfma(A, B, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    const int gy = y0 + wave * NT + t;
    if (gy < a.H && gx < a.W && oc < hc) {
      const size_t p = (size_t)(n * a.H + gy) * a.W + gx;
      const float4 b = a.head_b ? *reinterpret_cast<const float4*>(a.head_b + oc)
                                : make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // 16-byte aligned
      *reinterpret_cast<float4*>(a.head_y + p * hc + oc) =
          make_float4(h[0] + b.x, h[1] + b.y, h[2] + b.z, h[3] + b.w);
    }
  }
}

// What follows a tile's rounded outputs q: the 1x1 head, the 2x2 pool.
template <int MT, int NT, bool HEAD, bool POOL>
__device__ inline void conv_after(const ConvArgs& a, const bf16x4 (&q)[MT][NT], int n, int y0,
                                  int x0, int cb, int wave, int lane) {
  const int gx = x0 + (lane & 15);
  if constexpr (HEAD) conv_head<NT>(a, q, n, y0, x0, wave, lane);
  if constexpr (POOL) {
    // Rows y0 + NT wave + t pair as (t, t + 1) for even t (y0 and NT wave
    // are even); columns pair as lanes (l, l ^ 1).  The even lane of a pair
    // sums (top left, top right, bottom left, bottom right) in the order
    // of pool2_fwd_v8_kernel.  H and W are even, so a pooled pixel lies in
    // bounds exactly when its top-left input pixel does.
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int co = cb + m * 16 + (lane >> 4) * 4;
#pragma unroll
      for (int t = 0; t < NT; t += 2) {
        bf16x4 r0, r1;
        {
          int2 u0 = *reinterpret_cast<const int2*>(&q[m][t]);
          int2 u1 = *reinterpret_cast<const int2*>(&q[m][t + 1]);
          u0.x = __shfl_xor(u0.x, 1);
          u0.y = __shfl_xor(u0.y, 1);
          u1.x = __shfl_xor(u1.x, 1);
          u1.y = __shfl_xor(u1.y, 1);
          r0 = *reinterpret_cast<const bf16x4*>(&u0);
          r1 = *reinterpret_cast<const bf16x4*>(&u1);
        }
        const int gy = y0 + wave * NT + t;
        if ((lane & 1) == 0 && gy < a.H && gx < a.W && co < a.Cout) {
          bf16x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = (__bf16)(0.25f * ((float)q[m][t][i] + (float)r0[i] + (float)q[m][t + 1][i] +
                                     (float)r1[i]));
          const size_t pp = ((size_t)(n * (a.H >> 1) + (gy >> 1)) * (a.W >> 1) + (gx >> 1)) * a.Cout;
          *reinterpret_cast<bf16x4*>(a.pool_y + pp + co) = o;
        }
      }
    }
  }
}

// The epilogue of a block's tile: lane holds channels cb + 16m + 4(lane/16)
// + i of pixel (y0 + NT wave + t, x0 + lane%16).  HEAD: then the 1x1 head.
template <int MT, int NT, bool HEAD>
__device__ inline void conv_epilogue(const ConvArgs& a, const f32x4 (&acc)[MT][NT], int n, int y0,
                                     int x0, int cb, int wave, int lane) {
  const int gx = x0 + (lane & 15);
  bf16x4 q[MT][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int gy = y0 + wave * NT + t;
    const size_t p = (size_t)(n * a.H + gy) * a.W + gx;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int co = cb + m * 16 + (lane >> 4) * 4;
      q[m][t] = bf16x4{};
      if (gy < a.H && gx < a.W && co < a.Cout)
        q[m][t] = store_out4<HEAD>(a, p * a.Cout + co, co, acc[m][t]);
    }
  }
  if constexpr (HEAD) conv_head<NT>(a, q, n, y0, x0, wave, lane);
}

// Forward (and dgrad) convolution.  Block = 4 waves; each wave owns 32 pixels
// x 16*NT output channels as 2 x NT MFMA accumulators.
template <int TAPS, int NT>
__global__ void __launch_bounds__(256) conv_fwd_kernel(ConvArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int P = a.N * a.H * a.W;
  const int pb = (blockIdx.x * 4 + wave) * 32;
  const int cb = blockIdx.y * 16 * NT;
  const int K = a.K, Cin = a.Cin;
  int pn[2], py[2], px[2];
  bool pv[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int p = pb + r * 16 + (lane & 15);
    pv[r] = p < P;
    const int pp = pv[r] ? p : 0;
    px[r] = pp % a.W;
    py[r] = (pp / a.W) % a.H;
    pn[r] = pp / (a.W * a.H);
  }
  f32x4 acc[2][NT];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int ksteps = (K + 31) / 32;
  for (int ks = 0; ks < ksteps; ++ks) {
    const int k0 = ks * 32 + (lane >> 4) * 8;
    const bool kv = k0 < K;
    const int tap = kv ? k0 / Cin : 0;
    const int ci0 = kv ? k0 - tap * Cin : 0;
    const int dy = TAPS == 9 ? tap / 3 - 1 : 0;
    const int dx = TAPS == 9 ? tap % 3 - 1 : 0;
    bf16x8 A[2], B[NT];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int yy = py[r] + dy, xx = px[r] + dx;
      const bool ok = kv && pv[r] && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W;
      A[r] = ok ? load8(a.x + ((size_t)(pn[r] * a.H + yy) * a.W + xx) * Cin + ci0) : zero8();
    }
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      const int co = cb + c * 16 + (lane & 15);
      B[c] = (kv && co < a.Cout) ? load8(a.w + (size_t)co * K + k0) : zero8();
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < NT; ++c) acc[r][c] = mfma(A[r], B[c], acc[r][c]);
  }
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      const int co = cb + c * 16 + (lane & 15);
      if (co >= a.Cout) continue;
      const float bv = a.bias ? a.bias[co] : 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = pb + r * 16 + (lane >> 4) * 4 + i;
        if (p >= P) continue;
        float v = acc[r][c][i] + bv;
        const size_t o = (size_t)p * a.Cout + co;
        if (a.res) v += (float)a.res[o];
        if (a.relu) v = v > 0.0f ? v : 0.0f;
        if (a.y_f) a.y_f[o] = v;
        else a.y_bf[o] = (__bf16)v;
      }
    }
}

// Tile width of the LDS-staged convolutions, and LDS bf16 per patch pixel
// (32 channels + 8: spreads the banks).
constexpr int kTW = 16;
constexpr int kPS = 40;

// Forward (and dgrad) convolution for Cin and Cout multiples of 32, staged
// through LDS.  A block owns a 16 (x) by 4*NT (y) pixel tile of one image and
// 16*MT output channels.  Per 32-channel chunk of the input it stages the
// tile's input patch with a 1-pixel halo (TAPS = 9) and the chunk's weights
// for every tap; output channels are the MFMA's M operand (A = weights),
// pixels its N operand (B = patch), so a lane ends with 4 consecutive
// channels of one pixel and stores them as one vector.  Wave w owns tile
// rows NT*w .. NT*w+NT-1 (one 16-pixel N tile each).  The next chunk's patch
// and weights are
// loaded into registers while the current chunk's MFMAs run (the global
// loads' latency hides behind them; LDS holds one chunk), and each patch row
// read from LDS once per column shift dx and used for the three row shifts
// dy (a wave's NT output rows need NT + 2 patch rows): per chunk and wave
// 3 (NT + 2) B reads and 9 MT A reads feed 9 MT NT MFMAs.
template <int TAPS, int MT, int NT, bool UPCAT = false, bool HEAD = false>
__global__ void __launch_bounds__(256, 2) conv_pf_kernel(ConvArgs a) {
  constexpr int kTH = 4 * NT;
  constexpr int HALO = TAPS == 9 ? 1 : 0;
  constexpr int PW = kTW + 2 * HALO, PH = kTH + 2 * HALO;
  constexpr int WS = TAPS * 32 + 8;  // LDS bf16 per output channel of the weight chunk
  constexpr int NPV = PH * PW * 4;             // 16-byte patch vectors per chunk
  constexpr int NWV = MT * 16 * TAPS * 4;      // 16-byte weight vectors per chunk
  constexpr int RP = (NPV + 255) / 256, RW = (NWV + 255) / 256;
  constexpr int NS = 2 * HALO + 1;             // column (and row) shifts
  __shared__ __bf16 patch[PH * PW * kPS];
  __shared__ __bf16 wl[MT * 16 * WS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_x = (a.W + kTW - 1) / kTW, tiles_y = (a.H + kTH - 1) / kTH;
  int b = blockIdx.x;
  const int tx = b % tiles_x;
  b /= tiles_x;
  const int ty = b % tiles_y;
  const int n = b / tiles_y;
  const int x0 = tx * kTW, y0 = ty * kTH;
  const int cb = blockIdx.y * MT * 16;
  const int Cin = a.Cin, K = a.K;
  bf16x8 rp[RP], rw[RW];
  auto gload = [&](int ci0) {
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      const int v = threadIdx.x + 256 * j;
      bf16x8 val = zero8();
      if (v < NPV) {
        const int pix = v >> 2, q = v & 3;
        const int py = pix / PW, px = pix % PW;
        const int gy = y0 + py - HALO, gx = x0 + px - HALO;
        if (gy >= 0 && gy < a.H && gx >= 0 && gx < a.W) {
          const __bf16* src;
          if (!UPCAT)
            src = a.x + ((size_t)(n * a.H + gy) * a.W + gx) * Cin + ci0;
          else if (ci0 < a.C1)  // upsampled half: pixel (gy/2, gx/2) of x
            src = a.x + ((size_t)(n * (a.H >> 1) + (gy >> 1)) * (a.W >> 1) + (gx >> 1)) * a.C1 + ci0;
          else
            src = a.x2 + ((size_t)(n * a.H + gy) * a.W + gx) * (Cin - a.C1) + (ci0 - a.C1);
          val = load8(src + q * 8);
        }
      }
      rp[j] = val;
    }
#pragma unroll
    for (int j = 0; j < RW; ++j) {
      const int v = threadIdx.x + 256 * j;
      bf16x8 val = zero8();
      if (v < NWV) {
        const int co = v / (TAPS * 4), r = v % (TAPS * 4);
        const int tap = r >> 2, q = r & 3;
        if (cb + co < a.Cout) val = load8(a.w + (size_t)(cb + co) * K + tap * Cin + ci0 + q * 8);
      }
      rw[j] = val;
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      const int v = threadIdx.x + 256 * j;
      if (v < NPV)
        *reinterpret_cast<bf16x8*>(&patch[(v >> 2) * kPS + (v & 3) * 8]) = rp[j];
    }
#pragma unroll
    for (int j = 0; j < RW; ++j) {
      const int v = threadIdx.x + 256 * j;
      if (v < NWV) {
        const int co = v / (TAPS * 4), r = v % (TAPS * 4);
        *reinterpret_cast<bf16x8*>(&wl[co * WS + (r >> 2) * 32 + (r & 3) * 8]) = rw[j];
      }
    }
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // the next chunk loads into registers during this chunk's MFMAs
  gload(0);
  lstore();
  __syncthreads();
  for (int ci0 = 0; ci0 < Cin; ci0 += 32) {
    const bool more = ci0 + 32 < Cin;
    if (more) gload(ci0 + 32);
#pragma unroll
    for (int dx = 0; dx < NS; ++dx) {
      bf16x8 B[NT + 2 * HALO];
#pragma unroll
      for (int r = 0; r < NT + 2 * HALO; ++r) {
        const int row = wave * NT + r, col = (lane & 15) + dx;
        B[r] = *reinterpret_cast<const bf16x8*>(&patch[(row * PW + col) * kPS + (lane >> 4) * 8]);
      }
#pragma unroll
      for (int dy = 0; dy < NS; ++dy) {
        const int tap = dy * NS + dx;
        bf16x8 A[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
          A[m] = *reinterpret_cast<const bf16x8*>(&wl[(m * 16 + (lane & 15)) * WS + tap * 32 +
                                                      (lane >> 4) * 8]);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[m][t] = mfma(A[m], B[t + dy], acc[m][t]);
      }
    }
    __syncthreads();
    if (more) {
      lstore();
      __syncthreads();
    }
  }
  conv_epilogue<MT, NT, HEAD>(a, acc, n, y0, x0, cb, wave, lane);
}

// The same convolution with persistent blocks: block (b, co) takes the tiles
// b, b + gridDim.x, ... of output-channel block co, and the register
// prefetch of the next input chunk runs across tile boundaries: while the
// last chunk of one tile is multiplied, the first chunk of the block's next
// tile is loaded.  A layer of one or two 32-channel chunks then hides its
// load latency behind MFMAs as a deep layer does, where one tile per block
// leaves every block waiting for its patch.  A single-chunk layer loads its
// weights once per block.  Three blocks per compute unit with 32 output
// channels per block (MT = 2): at most 168 VGPRs and 45 KB of LDS each.
//
// The address work is kept off the vector units, which issue it in the shadow
// of nothing (a step of 72 MFMAs per wave came with 460 other vector
// instructions and a branch per load and bounds check; level-0 layers spent
// as long issuing as waiting for memory): every access goes through a buffer
// whose base the scalar unit sets per tile, with a lane offset that never
// changes.  A row above the image gives an offset that wraps and a row below
// one past the buffer's end; both read zeros and store nothing, as the
// hardware checks each offset against the buffer's size, so only the tiles at
// the left and right edge compare columns.  The rows of one tile must span
// less than 2^31 bytes (tile_rows_fit).  A tile's residual (kEpiRes) or the
// backward pass's residual and mask (kEpiGrad, kEpiMask) are on their way while the next
// tile goes to LDS, or a row of them.
// Measured against the same loop with an address, a bounds check and a branch
// per load (us, at batch 16): 256^2, 32 -> 32 channels 40.1 -> 28.9 (4.6 TB/s),
// with residual and pool 65.2 -> 41.9; 128^2, 64 -> 64 38.2 -> 32.1; 64^2,
// 96 -> 96 21.3 -> 18.6; 256^2, [up2, skip] 96 -> 32 85.1 -> 73.9.
constexpr int kTileBlocksPerCU = 3;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// offset past the end of every buffer, also with a tile's offset added
constexpr uint32_t kOffNone = 0x80000000u;

// [base, base + bytes): reads past it give 0, writes past it are dropped
__device__ inline __amdgpu_buffer_rsrc_t tile_buffer(const void* base, long long bytes) {
  const int n = bytes < 0x7fffffffLL ? (int)bytes : 0x7fffffff;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, n, 0x00020000);
}

inline bool tile_rows_fit(const ConvArgs& a) {
  const long long c = std::max(a.Cin, 2 * a.Cout);  // an FP32 output counts twice
  return (long long)a.W * c * 2 * 20 < 0x7fffffffLL;
}

enum { kEpiPlain, kEpiRes, kEpiMask, kEpiGrad };  // + nothing, res, mask, gres (and mask)

template <int MT, int NT, bool UPCAT, bool HEAD, bool POOL, int EPI>
__global__ void __launch_bounds__(256, kTileBlocksPerCU) conv_tiles_kernel(ConvArgs a) {
  static_assert(MT == 2, "three blocks per CU fit 32 output channels per block");
  static_assert(!POOL || NT % 2 == 0, "the pool pairs a wave's rows");
  constexpr int kTH = 4 * NT;
  constexpr int PW = kTW + 2, PH = kTH + 2;
  constexpr int WS = 9 * 32 + 8;          // LDS bf16 per output channel of the weight chunk
  constexpr int NPV = PH * PW * 4;        // 16-byte patch vectors per chunk
  constexpr int NWV = MT * 16 * 9 * 4;    // 16-byte weight vectors per chunk
  constexpr int RP = (NPV + 255) / 256, RW = (NWV + 255) / 256;
  __shared__ __align__(16) __bf16 patch[PH * PW * kPS];
  __shared__ __align__(16) __bf16 wl[MT * 16 * WS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_x = (a.W + kTW - 1) / kTW, tiles_y = (a.H + kTH - 1) / kTH;
  const int total = a.N * tiles_x * tiles_y;
  int tile = blockIdx.x;
  if (tile >= total) return;  // uniform over the block
  const int cb = blockIdx.y * MT * 16;
  const int Cin = a.Cin, K = a.K;
  const bool reload_w = Cin > 32;  // one chunk: its weights stay in LDS
  // this thread's patch and weight vectors, in bytes from the tile's first
  // halo pixel (UPCAT: of the second input, and poh of the half-size first one)
  const int CS = UPCAT ? Cin - a.C1 : Cin, Wh = a.W >> 1;
  uint32_t po[RP], poh[RP], wo[RW];
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const int v = threadIdx.x + 256 * j, pix = v >> 2, py = pix / PW, px = pix % PW;
    po[j] = v < NPV ? (uint32_t)((py * a.W + px) * CS * 2 + (v & 3) * 16) : kOffNone;
    if (UPCAT)
      poh[j] = v < NPV ? (uint32_t)((((py + 1) >> 1) * Wh + ((px + 1) >> 1)) * a.C1 * 2 + (v & 3) * 16)
                       : kOffNone;
  }
#pragma unroll
  for (int j = 0; j < RW; ++j) {
    const int v = threadIdx.x + 256 * j, co = v / 36, r = v % 36;
    wo[j] = v < NWV ? (uint32_t)((co * K + (r >> 2) * Cin) * 2 + (r & 3) * 16) : kOffNone;
  }
  const __amdgpu_buffer_rsrc_t wbuf =
      tile_buffer(a.w + (size_t)cb * K, (long long)MT * 16 * K * 2);
  u32x4 rp[RP], rw[RW];
  auto gload = [&](int t, int ci0, bool wts) {
    const int tx = t % tiles_x, r = t / tiles_x;
    const int x0 = tx * kTW, y0 = (r % tiles_y) * kTH, n = r / tiles_y;
    const bool edge = x0 == 0 || x0 + kTW >= a.W;
    const bool half = UPCAT && ci0 < a.C1;
    // the buffer: the image's rows from the patch's first one on
    const int C = half ? a.C1 : CS, w = half ? Wh : a.W, h = half ? a.H >> 1 : a.H;
    const int sx = half ? x0 >> 1 : x0, sy = half ? y0 >> 1 : y0, c0 = UPCAT && !half ? ci0 - a.C1 : ci0;
    const int row0 = sy > 0 ? sy - 1 : 0;
    const __bf16* src = UPCAT && !half ? a.x2 : a.x;
    const long long row_bytes = (long long)w * C * 2;
    const __amdgpu_buffer_rsrc_t buf =
        tile_buffer(src + ((size_t)n * h + row0) * w * C, (h - row0) * row_bytes);
    const uint32_t toff =
        (uint32_t)((sy - 1 - row0) * (int)row_bytes + (sx - 1) * C * 2 + c0 * 2);
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      uint32_t o = (half ? poh[j] : po[j]) + toff;
      if (edge) {
        const int px = ((threadIdx.x + 256 * j) >> 2) % PW;
        if ((uint32_t)(x0 - 1 + px) >= (uint32_t)a.W) o = kOffNone;
      }
      rp[j] = __builtin_amdgcn_raw_buffer_load_b128(buf, o, 0, 0);
    }
    if (wts) {
#pragma unroll
      for (int j = 0; j < RW; ++j)
        rw[j] = __builtin_amdgcn_raw_buffer_load_b128(wbuf, wo[j] + (uint32_t)ci0 * 2, 0, 0);
    }
  };
  auto lstore = [&](bool wts) {
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      const int v = threadIdx.x + 256 * j;
      if (v < NPV) *reinterpret_cast<u32x4*>(&patch[(v >> 2) * kPS + (v & 3) * 8]) = rp[j];
    }
    if (wts) {
#pragma unroll
      for (int j = 0; j < RW; ++j) {
        const int v = threadIdx.x + 256 * j;
        if (v < NWV) {
          const int co = v / 36, r2 = v % 36;
          *reinterpret_cast<u32x4*>(&wl[co * WS + (r2 >> 2) * 32 + (r2 & 3) * 8]) = rw[j];
        }
      }
    }
  };
  // this lane's outputs, in bytes (BF16) from the tile's first pixel
  const uint32_t lane_out =
      (uint32_t)((wave * NT * a.W + (lane & 15)) * a.Cout * 2 + (lane >> 4) * 8);
  gload(tile, 0, true);
  lstore(true);
  __syncthreads();
  for (;;) {
    const int tx = tile % tiles_x, r = tile / tiles_x;
    const int n = r / tiles_y, y0 = (r % tiles_y) * kTH, x0 = tx * kTW;
    const size_t out0 = (((size_t)n * a.H + y0) * a.W + x0) * a.Cout + cb;
    const long long out_bytes = (((long long)(a.H - y0)) * a.W - x0) * a.Cout * 2 - cb * 2;
    const uint32_t lo = x0 + (lane & 15) < a.W ? lane_out : kOffNone;
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto load_row = [&](const __bf16* p, int t, u32x2 (&e)[MT][NT]) {
      const __amdgpu_buffer_rsrc_t buf = tile_buffer(p + out0, p ? out_bytes : 0);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        e[m][t] = __builtin_amdgcn_raw_buffer_load_b64(
            buf, lo + (uint32_t)(t * a.W * a.Cout * 2) + m * 32, 0, 0);
    };
    auto load_out = [&](const __bf16* p, u32x2 (&e)[MT][NT]) {
#pragma unroll
      for (int t = 0; t < NT; ++t) load_row(p, t, e);
    };
    for (int ci0 = 0;; ci0 += 32) {
      // the next (tile, chunk) of this block
      const bool last = ci0 + 32 >= Cin;
      const int nt = last ? tile + (int)gridDim.x : tile;
      if (nt < total) gload(nt, last ? 0 : ci0 + 32, reload_w);
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        bf16x8 B[NT + 2];
#pragma unroll
        for (int r = 0; r < NT + 2; ++r) {
          const int row = wave * NT + r, col = (lane & 15) + dx;
          B[r] = *reinterpret_cast<const bf16x8*>(&patch[(row * PW + col) * kPS + (lane >> 4) * 8]);
        }
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const int tap = dy * 3 + dx;
          bf16x8 A[MT];
#pragma unroll
          for (int m = 0; m < MT; ++m)
            A[m] = *reinterpret_cast<const bf16x8*>(&wl[(m * 16 + (lane & 15)) * WS + tap * 32 +
                                                        (lane >> 4) * 8]);
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[m][t] = mfma(A[m], B[t + dy], acc[m][t]);
        }
      }
      if (last) break;
      __syncthreads();
      lstore(reload_w);
      __syncthreads();
    }
    u32x2 e0[MT][NT], e1[MT][NT];
    constexpr bool rowwise = EPI == kEpiGrad && NT > 2;
    if (EPI == kEpiRes) load_out(a.res, e0);
    if (EPI == kEpiGrad && !rowwise) load_out(a.gres, e0);
    if ((EPI == kEpiGrad && !rowwise) || EPI == kEpiMask) load_out(a.mask, e1);
    const bool next = tile + (int)gridDim.x < total;  // uniform over the block
    if (next) {
      __syncthreads();
      lstore(reload_w);
    }
    // The residual and the mask of the backward pass with 16 x 16 tiles: a row of
    // the wave ahead, from here on.  Whole tiles of both beside the next tile's
    // registers spilled (52 bytes a thread; at batch 16, us with all rows before
    // the store to LDS / row by row: 128^2 64 -> 64 channels 48.9 / 39.7, 96 -> 128 104.8
    // / 89.2, 64^2 96 -> 96 21.0 / 18.0), and without the fences the compiler moves
    // them up.  (Row by row with 16 x 8 tiles: 32^2 512 -> 512 at batch 1 23.9 / 29.2.)
    if (rowwise) {
      __builtin_amdgcn_sched_barrier(0);
      load_row(a.gres, 0, e0);
      load_row(a.mask, 0, e1);
    }
    if (next) __syncthreads();
    // store_out4's steps
    bf16x4 q[MT][NT];
    float4 bias[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
      bias[m] = a.bias ? *reinterpret_cast<const float4*>(a.bias + cb + m * 16 + (lane >> 4) * 4)
                       : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const bool bf_out = !a.y_f && (!HEAD || a.y_bf);
    const __amdgpu_buffer_rsrc_t ybuf = tile_buffer(a.y_bf + out0, bf_out ? out_bytes : 0);
    const __amdgpu_buffer_rsrc_t fbuf = tile_buffer(a.y_f + out0, a.y_f ? 2 * out_bytes : 0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (rowwise) {
        if (t + 1 < NT) {
          load_row(a.gres, t + 1, e0);
          load_row(a.mask, t + 1, e1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const uint32_t o = lo + (uint32_t)(t * a.W * a.Cout * 2) + m * 32;
        float v[4] = {acc[m][t][0] + bias[m].x, acc[m][t][1] + bias[m].y,
                      acc[m][t][2] + bias[m].z, acc[m][t][3] + bias[m].w};
        if (EPI == kEpiRes) {
          const bf16x4 res = __builtin_bit_cast(bf16x4, e0[m][t]);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] += (float)res[i];
        }
        if (a.relu) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) q[m][t][i] = (__bf16)v[i];
        if (EPI == kEpiGrad) {
          const bf16x4 gr = __builtin_bit_cast(bf16x4, e0[m][t]);
#pragma unroll
          for (int i = 0; i < 4; ++i) q[m][t][i] = (__bf16)((float)q[m][t][i] + (float)gr[i]);
        }
        if (EPI == kEpiGrad || EPI == kEpiMask) {
          const bf16x4 mk = __builtin_bit_cast(bf16x4, e1[m][t]);
          if (EPI == kEpiMask || a.mask) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              q[m][t][i] = (float)mk[i] > 0.0f ? q[m][t][i] : (__bf16)0.0f;
          }
        }
        if (bf_out)
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, q[m][t]), ybuf, o, 0, 0);
        if (a.y_f) {
          const float4 f = make_float4(v[0], v[1], v[2], v[3]);
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f), fbuf,
                                                 lo == kOffNone ? kOffNone : 2 * o, 0, 0);
        }
      }
    }
    conv_after<MT, NT, HEAD, POOL>(a, q, n, y0, x0, cb, wave, lane);
    tile += (int)gridDim.x;
    if (tile >= total) break;
  }
}

// 3x3 convolution of an 8-channel input (the network's first layer), staged
// through LDS.  K = 9 taps x 8 channels = 72, padded to three MFMA k-steps of
// 32: k-step j takes taps 4j .. 4j+3 (lane group q = lane/16 reads tap 4j+q,
// zero past tap 8), each tap's 8 channels one 16-byte patch vector.  Output
// channels are the M operand and pixels the N operand, as in conv_pf_kernel,
// whose epilogue this shares: a lane stores 4 consecutive channels at once.
template <int MT, int NT>
__global__ void __launch_bounds__(256) conv_c8_kernel(ConvArgs a) {
  constexpr int kTH = 4 * NT, PW = kTW + 2, PH = kTH + 2;
  constexpr int KP = 96 + 8;  // LDS bf16 per output channel of the weights (72 used, padded)
  __shared__ bf16x8 patch[PH * PW];
  __shared__ __bf16 wl[MT * 16 * KP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_x = (a.W + kTW - 1) / kTW, tiles_y = (a.H + kTH - 1) / kTH;
  int b = blockIdx.x;
  const int tx = b % tiles_x;
  b /= tiles_x;
  const int ty = b % tiles_y;
  const int n = b / tiles_y;
  const int x0 = tx * kTW, y0 = ty * kTH;
  const int cb = blockIdx.y * MT * 16;
  for (int v = threadIdx.x; v < PH * PW; v += 256) {
    const int py = v / PW, px = v % PW;
    const int gy = y0 + py - 1, gx = x0 + px - 1;
    bf16x8 val = zero8();
    if (gy >= 0 && gy < a.H && gx >= 0 && gx < a.W)
      val = load8(a.x + ((size_t)(n * a.H + gy) * a.W + gx) * 8);
    patch[v] = val;
  }
  for (int v = threadIdx.x; v < MT * 16 * 12; v += 256) {  // 12 taps of 8 per channel
    const int co = v / 12, tap = v % 12;
    bf16x8 val = zero8();
    if (tap < 9 && cb + co < a.Cout) val = load8(a.w + (size_t)(cb + co) * 72 + tap * 8);
    *reinterpret_cast<bf16x8*>(&wl[co * KP + tap * 8]) = val;
  }
  __syncthreads();
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int q = lane >> 4;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int tap = 4 * j + q;
    const int dy = tap < 9 ? tap / 3 : 0, dx = tap < 9 ? tap % 3 : 0;
    bf16x8 A[MT], B[NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
      A[m] = *reinterpret_cast<const bf16x8*>(&wl[(m * 16 + (lane & 15)) * KP + tap * 8]);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bf16x8 v = patch[(wave * NT + t + dy) * PW + (lane & 15) + dx];
      B[t] = tap < 9 ? v : zero8();
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[m][t] = mfma(A[m], B[t], acc[m][t]);
  }
  conv_epilogue<MT, NT, false>(a, acc, n, y0, x0, cb, wave, lane);
}

// dgrad weights: Wf[ci][tap'*Cout + co] = W[co][(TAPS-1-tap')*Cin + ci]
__global__ void flip_weights_kernel(const __bf16* __restrict__ w, __bf16* wf, int Cin, int Cout,
                                    int taps) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = Cin * Cout * taps;
  if (i >= n) return;
  const int ci = i / (taps * Cout);
  const int rem = i % (taps * Cout);
  const int tp = rem / Cout, co = rem % Cout;
  wf[i] = w[(size_t)co * taps * Cin + (taps - 1 - tp) * Cin + ci];
}

struct WgradArgs {
  const __bf16* __restrict__ x;  // [P][Cin] input of the convolution
  const __bf16* __restrict__ g;  // [P][Cout] gradient of its output
  float* part;                   // [splits][Cout][K]
  int N, H, W, Cin, Cout, K, taps;
  int chunk;                     // pixels per split (multiple of 32)
};

// One wave per block: a 32 (co) x 32 (k) tile of dW over one pixel range.
__global__ void __launch_bounds__(64) conv_wgrad_kernel(WgradArgs a) {
  __shared__ __bf16 Gs[32][32 + 8];  // [pixel][co]
  __shared__ __bf16 Xs[32][32 + 8];  // [pixel][k]
  const int lane = threadIdx.x;
  const int P = a.N * a.H * a.W;
  const int cb = blockIdx.x * 32, kb = blockIdx.y * 32;
  const int p_begin = blockIdx.z * a.chunk;
  const int p_end = min(P, p_begin + a.chunk);
  f32x4 acc[2][2];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int p0 = p_begin; p0 < p_end; p0 += 32) {
    // stage: 32 pixels x 4 groups of 8 channels, for G and for the tap-shifted X
    for (int t = lane; t < 128; t += 64) {
      const int pi = t >> 2, grp = t & 3;
      const int p = p0 + pi;
      const int co = cb + grp * 8;
      bf16x8 gv = zero8();
      if (p < p_end && co < a.Cout) gv = load8(a.g + (size_t)p * a.Cout + co);
      const int k0 = kb + grp * 8;
      bf16x8 xv = zero8();
      if (p < p_end && k0 < a.K) {
        const int tap = k0 / a.Cin, ci0 = k0 - tap * a.Cin;
        const int dy = a.taps == 9 ? tap / 3 - 1 : 0, dx = a.taps == 9 ? tap % 3 - 1 : 0;
        const int xx = p % a.W, yy = (p / a.W) % a.H, nn = p / (a.W * a.H);
        const int y2 = yy + dy, x2 = xx + dx;
        if (y2 >= 0 && y2 < a.H && x2 >= 0 && x2 < a.W)
          xv = load8(a.x + ((size_t)(nn * a.H + y2) * a.W + x2) * a.Cin + ci0);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        Gs[pi][grp * 8 + i] = gv[i];
        Xs[pi][grp * 8 + i] = xv[i];
      }
    }
    __syncthreads();
    // A[m = co][kk = pixel], B[kk = pixel][n = k]
    bf16x8 A[2], B[2];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int i = 0; i < 8; ++i) A[r][i] = Gs[(lane >> 4) * 8 + i][r * 16 + (lane & 15)];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) B[c][i] = Xs[(lane >> 4) * 8 + i][c * 16 + (lane & 15)];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[r][c] = mfma(A[r], B[c], acc[r][c]);
    __syncthreads();
  }
  float* out = a.part + (size_t)blockIdx.z * a.Cout * a.K;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int co = cb + r * 16 + (lane >> 4) * 4 + i;
        const int k = kb + c * 16 + (lane & 15);
        if (co < a.Cout && k < a.K) out[(size_t)co * a.K + k] = acc[r][c][i];
      }
}

// Weight gradient for Cin and Cout multiples of 32, TAPS = 9, staged through
// LDS: dW[co][tap*Cin + ci] = sum_p g[p][co] x[p + tap][ci]; its last blocks
// take the partials of the bias gradient sum_p g[p][co] (bias_partial).
// The reduction runs over pixels, so both MFMA operands need 8 pixels of one
// channel per lane, while the tiles lie pixel by pixel: G [8 rows][16 pixels]
// [32 co] and X [10 rows][18 pixels][32 ci] (the 1-pixel halo).  They are staged
// as they lie, and ds_read_b64_tr_b16 transposes while reading: each 16 lanes
// give four pixels x 16 channels, lane j receives channel j of the four.  A tap's
// shift is then only an address, also for odd columns.
// The order of the sums is part of the results: FP32 sums in another order are
// as accurate, but Adam divides each gradient by its own size, so that from a
// difference of 1e-7 a few steps of training lead to other BF16 weights.  An
// element's products are added two rows of 16 pixels (one MFMA) after the other, tile
// by tile of 16 x 8 pixels, over a range of tiles that follows from the shape and
// the partials given; no tile shape, block shape or staging may change that.
// A block owns 32 output channels x 32 input channels x all 9 taps; a wave the
// taps of one column shift and 16 input channels.  It goes down the rows of X: the
// two rows from row j on serve the taps (s, dy) with 2 s + dy = j, so every pair of
// rows is read once (17 fragments for 24 products; a wave per 16 x 16 channels and
// nine taps would read 31 for 36).  While a tile is multiplied, the next one comes
// from memory into registers and from there into the other half of LDS: one
// barrier a tile.  Off-image pixels are loaded from the image's first pixel and
// stored as zeros, so no load depends on a branch.
// A layer's launches, bias gradient and sums of the partials included, in us at
// batch 16: tiles stored transposed, without loads ahead and with launches for
// the bias / these with 3 waves of 32 input channels / 6 of 16 / 6 and two halves
// of LDS: 256^2 32 -> 32 channels 95.8 / 53.1 / 48.8 / 49.8, 256^2 96 -> 32 264 / 117 / 105
// / 102, 128^2 64 -> 64 101 / 48.7 / 46.8 / 41.1, 128^2 160 -> 64 221 / 98.7 / 91.6 /
// 83.5, 64^2 224 -> 96 125 / 56.3 / 52.3 / 50.5, 32^2 128 -> 128 48.2 / 24.4 / 23.2 / 20.0
// (the last with its channel blocks dealt out, see wgrad_lds).
// (The bias blocks first in the grid: 128^2 64 -> 64 51.0.)
constexpr int kWgTW = 16, kWgTH = 8, kWgPix = kWgTW * kWgTH;
constexpr int kWgXW = kWgTW + 2, kWgXPix = kWgXW * (kWgTH + 2);
constexpr int kWgThreads = 384;  // a wave per column shift and 16 input channels
constexpr int kWgS = 32 + 8;     // halfwords per pixel in LDS; 16 pixels cover the banks evenly
constexpr int kWgHalf = (kWgPix + kWgXPix) * kWgS;  // a tile's, 24640 bytes

struct WgArgs {
  // the input: x [N][H][W][Cin], or (C1 > 0) its channels below C1 from x
  // [N][H/2][W/2][C1], read at (y/2, x/2), and the others from x2
  const __bf16* __restrict__ x;
  const __bf16* __restrict__ x2;
  int C1;
  const __bf16* __restrict__ g;
  float* part;  // [splits][Cout*K]
  int N, H, W, Cin, Cout, K;
  int tiles_x, tiles_y, tiles;
  int tiles_per_split;
  int xcds;
  int blocks;            // of the weight gradient; those after it sum the bias gradient
  float* bias_part;      // [ranges of bias_rows pixels][Cout]
  int bias_rows;
};

// bias_grad_v8_kernel's partial of range b of rows_per_block pixels, 32 channels
// from c0 on, by a block of NT threads: the same sums in the same order
// (thread t takes the work of that kernel's threads t, t + NT, ... of these
// channels).  acc: 8192 floats of LDS.
template <int NT>
__device__ inline void bias_partial(const __bf16* __restrict__ g, float* part, int P, int C,
                                    int rows_per_block, int b, int c0, float* acc) {
  const int groups = 1024 / (C / 8);
  const int p0 = b * rows_per_block, p1 = min(P, p0 + rows_per_block);
  for (int v = threadIdx.x; v < 4 * groups; v += NT) {
    const int r = v >> 2;
    const __bf16* gc = g + c0 + 8 * (v & 3);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int p = p0 + r;
    for (; p + 7 * groups < p1; p += 8 * groups) {
      bf16x8 x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = load8(gc + (size_t)(p + u * groups) * C);
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] += (float)x[u][k];
    }
    for (; p < p1; p += groups) {
      const bf16x8 x = load8(gc + (size_t)p * C);
#pragma unroll
      for (int k = 0; k < 8; ++k) s[k] += (float)x[k];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[v * 8 + k] = s[k];
  }
  __syncthreads();
  for (int n = groups; n > 1;) {
    const int h = (n + 1) / 2;
    for (int i = threadIdx.x; i < (n - h) * 32; i += NT) acc[i] += acc[h * 32 + i];
    __syncthreads();
    n = h;
  }
  if (threadIdx.x < 32) part[(size_t)b * C + c0 + threadIdx.x] = acc[threadIdx.x];
}

// 8 pixels of one channel: p = this lane's 4 channels of its pixel of the
// first four
__device__ inline bf16x8 read_pixels8(const __bf16* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * kWgS));
  return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

__global__ void __launch_bounds__(kWgThreads) wgrad_lds_kernel(WgArgs a) {
  constexpr int NT = kWgThreads;
  constexpr int RG = (kWgPix * 4 + NT - 1) / NT, RX = (kWgXPix * 4 + NT - 1) / NT;
  __shared__ __align__(16) float lds[kWgHalf];  // two halves, or bias_partial's floats
  static_assert(kWgHalf >= 8192, "bias_partial's floats");
  __bf16* gt = reinterpret_cast<__bf16*>(lds);
  __bf16* xt = gt + kWgPix * kWgS;
  if ((int)blockIdx.x >= a.blocks) {
    const int b = (int)blockIdx.x - a.blocks, nc = a.Cout / 32;
    bias_partial<NT>(a.g, a.bias_part, a.N * a.H * a.W, a.Cout, a.bias_rows, b / nc, b % nc * 32,
                     lds);
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, dx = wave % 3, cw = wave / 3 * 16;
  const int Cin = a.Cin, Cout = a.Cout;
  // Workgroups go round-robin over the 8 XCDs: the channel blocks of one
  // range of tiles, which read the same g and x, follow each other on one XCD
  // and share its L2 (training step: 96 -> 96 channels at 64^2 31 -> 23.5 us)
  // (a.xcds = 8), unless that leaves the XCDs with unequal work (a.xcds = 1; wgrad_lds)
  const int nco = Cout / 32, nch = nco * (Cin / 32), seq = (int)blockIdx.x / a.xcds;
  const int split = seq / nch * a.xcds + (int)blockIdx.x % a.xcds, ch = seq % nch;
  const int cb = ch % nco * 32, ci0 = ch / nco * 32;
  const int t_begin = split * a.tiles_per_split;
  const int t_end = min(a.tiles, t_begin + a.tiles_per_split);
  if (t_begin >= t_end) return;  // uniform over the block
  // where this block's input channels lie
  const int up = ci0 < a.C1 ? 1 : 0;
  const __bf16* src = a.C1 > 0 && !up ? a.x2 : a.x;
  const int srcH = a.H >> up, srcW = a.W >> up;
  const int srcC = up ? a.C1 : Cin - a.C1, srcc = up ? ci0 : ci0 - a.C1;
  f32x4 acc[3][2];  // [tap row][half of the output channels]
#pragma unroll
  for (int dy = 0; dy < 3; ++dy)
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[dy][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 rg[RG], rx[RX];
  uint32_t okg = 0, okx = 0;
  auto gload = [&](int t) {
    const int tx = t % a.tiles_x, ty = (t / a.tiles_x) % a.tiles_y;
    const int n = t / (a.tiles_x * a.tiles_y);
    const int x0 = tx * kWgTW, y0 = ty * kWgTH;
    const __bf16* gi = a.g + (size_t)n * a.H * a.W * Cout + cb;
    const __bf16* xi = src + (size_t)n * srcH * srcW * srcC + srcc;
    okg = okx = 0;
#pragma unroll
    for (int j = 0; j < RG; ++j) {
      const int v = threadIdx.x + NT * j, pix = v >> 2, q = v & 3;
      const int gy = y0 + pix / kWgTW, gx = x0 + pix % kWgTW;
      const bool ok = v < kWgPix * 4 && gy < a.H && gx < a.W;
      okg |= ok ? 1u << j : 0u;
      rg[j] = load8(gi + (ok ? ((size_t)gy * a.W + gx) * Cout : 0) + q * 8);
    }
#pragma unroll
    for (int j = 0; j < RX; ++j) {
      const int v = threadIdx.x + NT * j, pix = v >> 2, q = v & 3;
      const int gy = y0 + pix / kWgXW - 1, gx = x0 + pix % kWgXW - 1;
      const bool ok = v < kWgXPix * 4 && gy >= 0 && gy < a.H && gx >= 0 && gx < a.W;
      okx |= ok ? 1u << j : 0u;
      rx[j] = load8(xi + (ok ? ((size_t)(gy >> up) * srcW + (gx >> up)) * srcC : 0) + q * 8);
    }
  };
  // into the half of LDS from halfword o on
  auto lstore = [&](int o) {
#pragma unroll
    for (int j = 0; j < RG; ++j) {
      const int v = threadIdx.x + NT * j;
      if (v < kWgPix * 4)
        *reinterpret_cast<bf16x8*>(&gt[o + (v >> 2) * kWgS + (v & 3) * 8]) =
            okg >> j & 1 ? rg[j] : zero8();
    }
#pragma unroll
    for (int j = 0; j < RX; ++j) {
      const int v = threadIdx.x + NT * j;
      if (v < kWgXPix * 4)
        *reinterpret_cast<bf16x8*>(&xt[o + (v >> 2) * kWgS + (v & 3) * 8]) =
            okx >> j & 1 ? rx[j] : zero8();
    }
  };
  // An MFMA's 32 pixels are two rows of 16; lane group lane/16 holds 8 of them:
  // row group/2, columns 8 (group % 2) on.  This lane's pixel of the first 4 of
  // the 8, and its 4 channels:
  const int grp = lane >> 4, p4 = (lane & 15) >> 2, ch0 = (lane & 3) * 4;
  const __bf16* gl = &gt[(grp * 8 + p4) * kWgS + ch0];
  const __bf16* xl = &xt[((grp >> 1) * kWgXW + (grp & 1) * 8 + p4 + dx) * kWgS + cw + ch0];
  gload(t_begin);
  lstore(0);
  int o = 0;
  for (int t = t_begin; t < t_end; ++t) {
    // tile t is in LDS, and the other half is no longer read
    __syncthreads();
    if (t + 1 < t_end) gload(t + 1);
    bf16x8 B[3];  // the pair of X rows from row 2 s + dy on
#pragma unroll
    for (int s = 0; s < kWgTH / 2; ++s) {
      bf16x8 A[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) A[m] = read_pixels8(gl + o + s * 32 * kWgS + m * 16);
#pragma unroll
      for (int dy = 0; dy < 3; ++dy) {
        if (s > 0 && dy == 0)
          B[0] = B[2];  // read as the last pair of the step before
        else
          B[dy] = read_pixels8(xl + o + (2 * s + dy) * kWgXW * kWgS);
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[dy][m] = mfma(A[m], B[dy], acc[dy][m]);
      }
    }
    o ^= kWgHalf;
    if (t + 1 < t_end) lstore(o);
  }
  float* out = a.part + (size_t)split * Cout * a.K;
  const int co0 = cb + (lane >> 4) * 4, k0 = ci0 + cw + (lane & 15);
#pragma unroll
  for (int dy = 0; dy < 3; ++dy)
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        out[(size_t)(co0 + m * 16 + i) * a.K + (dy * 3 + dx) * Cin + k0] = acc[dy][m][i];
}

// dW[i] = sum over splits of part[k][i] in a fixed order (deterministic):
// 8 interleaved slices of k, each summed in ascending k, then the slice sums
// in slice order.  32 outputs x 8 slices per block keep the loads coalesced
// and give every output 8 independent chains.
constexpr int kRedSlices = 8;

// db[c0 .. c0 + 7] from the bias partials part [nb][C], by a block of 256
// threads: bias_reduce_kernel's sums in their order.  C >= 32.
__device__ inline void bias_reduce8(const float* __restrict__ part, float* db, int C, int nb,
                                    int c0) {
  __shared__ float acc[256 * 8];
  const int groups = 1024 / (C / 8), r = threadIdx.x;
  if (r < groups) {
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int b = r; b < nb; b += groups) {
      const float4* q = reinterpret_cast<const float4*>(part + (size_t)b * C + c0);
      const float4 v0 = q[0], v1 = q[1];
      s[0] += v0.x; s[1] += v0.y; s[2] += v0.z; s[3] += v0.w;
      s[4] += v1.x; s[5] += v1.y; s[6] += v1.z; s[7] += v1.w;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[r * 8 + k] = s[k];
  }
  __syncthreads();
  for (int n = groups; n > 1;) {
    const int h = (n + 1) / 2;
    for (int i = r; i < (n - h) * 8; i += 256) acc[i] += acc[h * 8 + i];
    __syncthreads();
    n = h;
  }
  if (r < 8) db[c0 + r] = acc[r];
}

__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float* __restrict__ part,
                                                           float* dw, int n, int splits,
                                                           const float* __restrict__ bias_part,
                                                           float* db, int C, int nb) {
  __shared__ float acc[kRedSlices][32];
  const int blocks = (n + 31) / 32;  // the ones after them: 8 channels of db each
  if ((int)blockIdx.x >= blocks) {
    bias_reduce8(bias_part, db, C, nb, ((int)blockIdx.x - blocks) * 8);
    return;
  }
  const int e = threadIdx.x & 31, sl = threadIdx.x >> 5;
  const int i = blockIdx.x * 32 + e;
  float s = 0.0f;
  if (i < n) {
    // eight loads in flight per iteration, added in ascending k as before
    int k = sl;
    for (; k + 7 * kRedSlices < splits; k += 8 * kRedSlices) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part[(size_t)(k + u * kRedSlices) * n + i];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; k < splits; k += kRedSlices) s += part[(size_t)k * n + i];
  }
  acc[sl][e] = s;
  __syncthreads();
  if (sl == 0 && i < n) {
    float t = 0.0f;
#pragma unroll
    for (int q = 0; q < kRedSlices; ++q) t += acc[q][e];
    dw[i] = t;
  }
}

// part[b][c] = sum of g[p][c] over block b's rows, in a fixed order: for
// C <= 256 thread t covers channel t % C and every (256/C)-th row from row
// t / C (coalesced: neighbouring threads read neighbouring channels), then
// the row-group sums are added in group order.
__global__ void __launch_bounds__(256) bias_grad_kernel(const __bf16* __restrict__ g, float* part,
                                                        int P, int C, int rows_per_block) {
  __shared__ float acc[256];
  const int t = threadIdx.x;
  const int p0 = blockIdx.x * rows_per_block;
  const int p1 = min(P, p0 + rows_per_block);
  if (C <= 256) {
    const int groups = 256 / C;
    const int c = t % C, r = t / C;
    float s = 0.0f;
    if (r < groups)
      for (int p = p0 + r; p < p1; p += groups) s += (float)g[(size_t)p * C + c];
    acc[t] = s;
    __syncthreads();
    if (t < C) {
      float u = 0.0f;
      for (int q = 0; q < groups; ++q) u += acc[q * C + t];
      part[(size_t)blockIdx.x * C + t] = u;
    }
  } else {
    for (int c = t; c < C; c += 256) {
      float s = 0.0f;
      for (int p = p0; p < p1; ++p) s += (float)g[(size_t)p * C + c];
      part[(size_t)blockIdx.x * C + c] = s;
    }
  }
}

// The same sums 8 channels per thread (C % 8 == 0, C <= 1024, g 16-byte
// aligned), 1024 threads per block: thread t covers channels 8 (t % C8) ..
// + 7 of every G-th row from row t / C8 (G = 1024 / C8 row groups), each
// load 16 bytes, eight rows in flight; then the G group sums are folded in
// LDS by halves (group r + h onto group r), a fixed order.
__device__ inline void fold_groups(float* acc, int t, int C8, int groups) {
  const int c8 = t % C8, r = t / C8;
  for (int n = groups; n > 1;) {
    const int h = (n + 1) / 2;  // groups [h, n) onto [0, n - h)
    if (r < n - h) {
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[(r * C8 + c8) * 8 + k] += acc[((r + h) * C8 + c8) * 8 + k];
    }
    __syncthreads();
    n = h;
  }
}

__global__ void __launch_bounds__(1024) bias_grad_v8_kernel(const __bf16* __restrict__ g,
                                                            float* part, int P, int C,
                                                            int rows_per_block) {
  __shared__ float acc[1024 * 8];
  const int t = threadIdx.x, C8 = C / 8, groups = 1024 / C8;
  const int c8 = t % C8, r = t / C8;
  const int p0 = blockIdx.x * rows_per_block;
  const int p1 = min(P, p0 + rows_per_block);
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (r < groups) {
    int p = p0 + r;
    for (; p + 7 * groups < p1; p += 8 * groups) {
      bf16x8 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = load8(g + (size_t)(p + u * groups) * C + 8 * c8);
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] += (float)v[u][k];
    }
    for (; p < p1; p += groups) {
      const bf16x8 v = load8(g + (size_t)p * C + 8 * c8);
#pragma unroll
      for (int k = 0; k < 8; ++k) s[k] += (float)v[k];
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) acc[t * 8 + k] = s[k];
  __syncthreads();
  fold_groups(acc, t, C8, groups);
  for (int c = t; c < C; c += 1024) part[(size_t)blockIdx.x * C + c] = acc[c];
}

// db[c] = sum over the nb block partials part[b][c] (C % 8 == 0, C <= 1024):
// one block of 1024 threads, thread t adds the partials b = t / C8, + G, ...
// of 8 channels (four in flight), then the groups fold as above.
__global__ void __launch_bounds__(1024) bias_reduce_kernel(const float* __restrict__ part,
                                                           float* db, int C, int nb) {
  __shared__ float acc[1024 * 8];
  const int t = threadIdx.x, C8 = C / 8, groups = 1024 / C8;
  const int c8 = t % C8, r = t / C8;
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (r < groups) {
    int b = r;
    for (; b + 3 * groups < nb; b += 4 * groups) {
      float4 v[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4* q = reinterpret_cast<const float4*>(part + (size_t)(b + u * groups) * C + 8 * c8);
        v[u][0] = q[0];
        v[u][1] = q[1];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s[0] += v[u][0].x; s[1] += v[u][0].y; s[2] += v[u][0].z; s[3] += v[u][0].w;
        s[4] += v[u][1].x; s[5] += v[u][1].y; s[6] += v[u][1].z; s[7] += v[u][1].w;
      }
    }
    for (; b < nb; b += groups) {
      const float4* q = reinterpret_cast<const float4*>(part + (size_t)b * C + 8 * c8);
      const float4 v0 = q[0], v1 = q[1];
      s[0] += v0.x; s[1] += v0.y; s[2] += v0.z; s[3] += v0.w;
      s[4] += v1.x; s[5] += v1.y; s[6] += v1.z; s[7] += v1.w;
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) acc[t * 8 + k] = s[k];
  __syncthreads();
  fold_groups(acc, t, C8, groups);
  for (int c = t; c < C; c += 1024) db[c] = acc[c];
}

__global__ void relu_bwd_kernel(const __bf16* __restrict__ y, const __bf16* __restrict__ g,
                                __bf16* out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = (float)y[i] > 0.0f ? g[i] : (__bf16)0.0f;
}

// 2x2 average pool, NHWC, H and W even
__global__ void pool2_fwd_kernel(const __bf16* __restrict__ x, __bf16* y, int N, int H, int W,
                                 int C) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2;
  const size_t n = (size_t)N * Ho * Wo * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const size_t q = i / C;
  const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho), nn = (int)(q / ((size_t)Wo * Ho));
  const size_t b = ((size_t)(nn * H + 2 * yo) * W + 2 * xo) * C + c;
  const float s = (float)x[b] + (float)x[b + C] + (float)x[b + (size_t)W * C] +
                  (float)x[b + (size_t)W * C + C];
  y[i] = (__bf16)(0.25f * s);
}

__global__ void pool2_bwd_kernel(const __bf16* __restrict__ gy, __bf16* gx, int N, int H, int W,
                                 int C) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t n = (size_t)N * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const size_t q = i / C;
  const int x = (int)(q % W), y = (int)((q / W) % H), nn = (int)(q / ((size_t)W * H));
  const int Ho = H / 2, Wo = W / 2;
  gx[i] = (__bf16)(0.25f * (float)gy[((size_t)(nn * Ho + y / 2) * Wo + x / 2) * C + c]);
}

// nearest x2 upsample of x [N][H][W][C] into channels [c_off, c_off+C) of
// y [N][2H][2W][Cy] (the first half of a concat)
__global__ void up2_fwd_kernel(const __bf16* __restrict__ x, __bf16* y, int N, int H, int W, int C,
                               int Cy, int c_off) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = 2 * H, Wo = 2 * W;
  const size_t n = (size_t)N * Ho * Wo * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const size_t q = i / C;
  const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho), nn = (int)(q / ((size_t)Wo * Ho));
  y[q * Cy + c_off + c] = x[((size_t)(nn * H + yo / 2) * W + xo / 2) * C + c];
}

__global__ void up2_bwd_kernel(const __bf16* __restrict__ gy, __bf16* gx, int N, int H, int W,
                               int C, int Cy, int c_off) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t n = (size_t)N * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  const size_t q = i / C;
  const int x = (int)(q % W), y = (int)((q / W) % H), nn = (int)(q / ((size_t)W * H));
  const int Wo = 2 * W;
  const size_t b = ((size_t)(nn * 2 * H + 2 * y) * Wo + 2 * x) * Cy + c_off + c;
  const float s = (float)gy[b] + (float)gy[b + Cy] + (float)gy[b + (size_t)Wo * Cy] +
                  (float)gy[b + (size_t)Wo * Cy + Cy];
  gx[i] = (__bf16)s;
}

// copy x [P][C] into channels [c_off, c_off+C) of y [P][Cy] (dir 0), or back (dir 1)
__global__ void channels_copy_kernel(const __bf16* __restrict__ src, __bf16* dst, size_t P, int C,
                                     int Cy, int c_off, int dir) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P * C) return;
  const size_t p = i / C;
  const int c = (int)(i % C);
  if (dir == 0) dst[p * Cy + c_off + c] = src[i];
  else dst[i] = src[p * Cy + c_off + c];
}

__global__ void add_kernel(const __bf16* __restrict__ a, const __bf16* __restrict__ b, __bf16* y,
                           size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  y[i] = (__bf16)((float)a[i] + (float)b[i]);
}

// The same element-wise kernels on 8 channels (16 bytes) per thread, used
// when every channel count and offset is a multiple of 8.
__device__ inline void store8(__bf16* p, bf16x8 v) { *reinterpret_cast<bf16x8*>(p) = v; }

__global__ void relu_bwd_v8_kernel(const __bf16* __restrict__ y, const __bf16* __restrict__ g,
                                   __bf16* out, size_t n8) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n8) return;
  const bf16x8 a = load8(y + 8 * i), b = load8(g + 8 * i);
  bf16x8 r;
#pragma unroll
  for (int k = 0; k < 8; ++k) r[k] = (float)a[k] > 0.0f ? b[k] : (__bf16)0.0f;
  store8(out + 8 * i, r);
}

__global__ void add_v8_kernel(const __bf16* __restrict__ a, const __bf16* __restrict__ b,
                              __bf16* y, size_t n8) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n8) return;
  const bf16x8 u = load8(a + 8 * i), v = load8(b + 8 * i);
  bf16x8 r;
#pragma unroll
  for (int k = 0; k < 8; ++k) r[k] = (__bf16)((float)u[k] + (float)v[k]);
  store8(y + 8 * i, r);
}

__global__ void pool2_fwd_v8_kernel(const __bf16* __restrict__ x, __bf16* y, int N, int H, int W,
                                    int C) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
  if (i >= (size_t)N * Ho * Wo * C8) return;
  const int c = (int)(i % C8) * 8;
  const size_t q = i / C8;
  const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho), nn = (int)(q / ((size_t)Wo * Ho));
  const size_t b = ((size_t)(nn * H + 2 * yo) * W + 2 * xo) * C + c;
  const bf16x8 v0 = load8(x + b), v1 = load8(x + b + C), v2 = load8(x + b + (size_t)W * C),
               v3 = load8(x + b + (size_t)W * C + C);
  bf16x8 r;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    r[k] = (__bf16)(0.25f * ((float)v0[k] + (float)v1[k] + (float)v2[k] + (float)v3[k]));
  store8(y + q * C + c, r);
}

__global__ void pool2_bwd_v8_kernel(const __bf16* __restrict__ gy, __bf16* gx, int N, int H,
                                    int W, int C) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  if (i >= (size_t)N * H * W * C8) return;
  const int c = (int)(i % C8) * 8;
  const size_t q = i / C8;
  const int x = (int)(q % W), y = (int)((q / W) % H), nn = (int)(q / ((size_t)W * H));
  const int Ho = H / 2, Wo = W / 2;
  const bf16x8 v = load8(gy + ((size_t)(nn * Ho + y / 2) * Wo + x / 2) * C + c);
  bf16x8 r;
#pragma unroll
  for (int k = 0; k < 8; ++k) r[k] = (__bf16)(0.25f * (float)v[k]);
  store8(gx + q * C + c, r);
}

__global__ void up2_fwd_v8_kernel(const __bf16* __restrict__ x, __bf16* y, int N, int H, int W,
                                  int C, int Cy, int c_off) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = 2 * H, Wo = 2 * W, C8 = C / 8;
  if (i >= (size_t)N * Ho * Wo * C8) return;
  const int c = (int)(i % C8) * 8;
  const size_t q = i / C8;
  const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho), nn = (int)(q / ((size_t)Wo * Ho));
  store8(y + q * Cy + c_off + c, load8(x + ((size_t)(nn * H + yo / 2) * W + xo / 2) * C + c));
}

// gate (or null): the result is zeroed where it is not positive (ReLU's
// backward on what was upsampled)
__global__ void up2_bwd_v8_kernel(const __bf16* __restrict__ gy, __bf16* gx,
                                  const __bf16* __restrict__ gate, int N, int H, int W, int C,
                                  int Cy, int c_off) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  if (i >= (size_t)N * H * W * C8) return;
  const int c = (int)(i % C8) * 8;
  const size_t q = i / C8;
  const int x = (int)(q % W), y = (int)((q / W) % H), nn = (int)(q / ((size_t)W * H));
  const int Wo = 2 * W;
  const size_t b = ((size_t)(nn * 2 * H + 2 * y) * Wo + 2 * x) * Cy + c_off + c;
  const bf16x8 v0 = load8(gy + b), v1 = load8(gy + b + Cy), v2 = load8(gy + b + (size_t)Wo * Cy),
               v3 = load8(gy + b + (size_t)Wo * Cy + Cy);
  bf16x8 r;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    r[k] = (__bf16)((float)v0[k] + (float)v1[k] + (float)v2[k] + (float)v3[k]);
  if (gate) {
    const bf16x8 y = load8(gate + q * C + c);
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = (float)y[k] > 0.0f ? r[k] : (__bf16)0.0f;
  }
  store8(gx + q * C + c, r);
}

// The gradient of an encoder stage's output y [N][H][W][C], before its ReLU:
// the pooled path's gp [N][H/2][W/2][C] spread over 2x2, plus the decoder's
// channels [c_off, c_off + C) of gu [N][H][W][Cu], zeroed where y is not
// positive.  The roundings of the four passes it replaces (pool, channel
// copy, sum, ReLU), which moved 2.6 times the bytes: memory bound, and at 16 x
// 256^2 x 32 channels 50 us (4.4 TB/s) against 128.
__global__ void skip_bwd_v8_kernel(const __bf16* __restrict__ gp, const __bf16* __restrict__ gu,
                                   const __bf16* __restrict__ y, __bf16* out, int N, int H, int W,
                                   int C, int Cu, int c_off) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  if (i >= (size_t)N * H * W * C8) return;
  const int c = (int)(i % C8) * 8;
  const size_t q = i / C8;
  const int px = (int)(q % W), py = (int)((q / W) % H), nn = (int)(q / ((size_t)W * H));
  const bf16x8 a = load8(gp + ((size_t)(nn * (H / 2) + py / 2) * (W / 2) + px / 2) * C + c);
  const bf16x8 b = load8(gu + q * Cu + c_off + c), v = load8(y + q * C + c);
  bf16x8 r;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const __bf16 p = (__bf16)(0.25f * (float)a[k]);
    const __bf16 s = (__bf16)((float)p + (float)b[k]);
    r[k] = (float)v[k] > 0.0f ? s : (__bf16)0.0f;
  }
  store8(out + q * C + c, r);
}

__global__ void channels_copy_v8_kernel(const __bf16* __restrict__ src, __bf16* dst, size_t P,
                                        int C, int Cy, int c_off, int dir) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int C8 = C / 8;
  if (i >= P * C8) return;
  const size_t p = i / C8;
  const int c = (int)(i % C8) * 8;
  if (dir == 0) store8(dst + p * Cy + c_off + c, load8(src + p * C + c));
  else store8(dst + p * C + c, load8(src + p * Cy + c_off + c));
}

// masked MSE: loss partials and d(loss)/dy = 2 (y - t) m / count
__global__ void mse_kernel(const float* __restrict__ y, const float* __restrict__ t,
                           const float* __restrict__ m, __bf16* g, float* part, size_t n,
                           float inv_count) {
  __shared__ float red[256];
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.0f;
  if (i < n) {
    const float mk = m ? m[i] : 1.0f;
    const float d = (y[i] - t[i]) * mk;
    l = d * d;
    g[i] = (__bf16)(2.0f * d * inv_count);
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam (Kingma & Ba 2015) on FP32 master weights; optional bf16 copy
// With wf, the rounded weight also goes to its place in the data gradient's
// flipped weights (flip_weights_kernel's layout), so the backward pass needs
// no flip of its own: w[co][t*Cin + ci] -> wf[ci][(taps-1-t)*Cout + co].
struct AdamStep {
  float lr, b1, b2, eps, c1, c2, wd;
};

__device__ inline float adam_update(const AdamStep& a, size_t i, float* w,
                                    const float* __restrict__ g, float* m, float* v, float wd) {
  const float gi = g[i] + wd * w[i];
  const float mi = a.b1 * m[i] + (1.0f - a.b1) * gi;
  const float vi = a.b2 * v[i] + (1.0f - a.b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
  w[i] = wi;
  return wi;
}

__global__ void adam_kernel(AdamStep a, float* w, const float* __restrict__ g, float* m, float* v,
                            __bf16* w_bf, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float wi = adam_update(a, i, w, g, m, v, a.wd);
  if (w_bf) w_bf[i] = (__bf16)wi;
}

// A convolution's weights, their two bf16 copies, and (nb > 0) its bias, which
// takes no weight decay: one launch per layer.
__global__ void adam_conv_kernel(AdamStep a, float* w, const float* __restrict__ g, float* m,
                                 float* v, __bf16* w_bf, __bf16* wf, int Cin, int Cout, int taps,
                                 float* b, const float* __restrict__ bg, float* bm, float* bv,
                                 int nb) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int k = taps * Cin;
  const size_t n = (size_t)k * Cout;
  if (i >= n) {
    if (i - n < (size_t)nb) adam_update(a, i - n, b, bg, bm, bv, 0.0f);
    return;
  }
  const float wi = adam_update(a, i, w, g, m, v, a.wd);
  w_bf[i] = (__bf16)wi;
  const int co = (int)i / k, rem = (int)i % k;
  const int t = rem / Cin, ci = rem % Cin;
  wf[(size_t)ci * taps * Cout + (size_t)(taps - 1 - t) * Cout + co] = (__bf16)wi;
}

// ---------------------------------------------------------- tiled inference
// The network's input and output on a whole map, in four launches a map where
// separate element-wise passes, window copies and crops took about 90 of 3 to 10
// us each (1000 x 700 cells: 1404 -> 1121 us).

// A map's array: element (x, y) at p[x sx + y sy].
struct MapIn {
  const float* p;
  long long sx, sy;
  __device__ float at(int x, int y) const { return p[x * sx + y * sy]; }
};
struct FlowMaps {
  MapIn h, d, mx, my;
};

__device__ inline float signed_log1p(float v, float scale) {
  const float s = (float)((0.0f < v) - (v < 0.0f));
  return (s * log1pf(fabsf(v))) * scale;
}

// features: height, its central differences (replicated at the edges) x slope,
// log1p(d) scale (d clamped at 0), signed log1p of the momentum, two zeros
__global__ void flow_features_kernel(FlowMaps m, float* f, int X, int Y, float slope, float scale) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)X * Y) return;
  const int x = (int)(i / Y), y = (int)(i % Y);
  const float xp = m.h.at(x + 1 < X ? x + 1 : x, y), xm = m.h.at(x > 0 ? x - 1 : x, y);
  const float yp = m.h.at(x, y + 1 < Y ? y + 1 : y), ym = m.h.at(x, y > 0 ? y - 1 : y);
  const float d = m.d.at(x, y);
  float4* o = reinterpret_cast<float4*>(f + 8 * i);
  o[0] = make_float4(m.h.at(x, y), (xp - xm) * slope, (yp - ym) * slope,
                     log1pf(d <= 0.0f ? 0.0f : d) * scale);
  o[1] = make_float4(signed_log1p(m.mx.at(x, y), scale), signed_log1p(m.my.at(x, y), scale), 0.0f,
                     0.0f);
}

// up to kJobs windows per launch, passed by value
constexpr int kJobs = 32;
struct WindowJobs {
  int wx[kJobs], wy[kJobs];  // the window's first cell
  int cx[kJobs], cy[kJobs];  // its core's first cell and sides
  int lx[kJobs], ly[kJobs];
};

// window k of feats [X][Y][8] into out[k] [tile][tile][8]
__global__ void window_copy_kernel(const float* __restrict__ feats, float* out, WindowJobs j,
                                   int Y, int tile) {
  const int k = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= tile * tile * 2) return;
  const int half = c & 1, p = c >> 1, x = p / tile, y = p % tile;
  const float4* src = reinterpret_cast<const float4*>(feats);
  reinterpret_cast<float4*>(out)[(size_t)k * tile * tile * 2 + c] =
      src[2 * ((size_t)(j.wx[k] + x) * Y + j.wy[k] + y) + half];
}

// windows to bf16, the height centred on its window's mean and scaled
__global__ void window_input_kernel(const float* __restrict__ xs, const float* __restrict__ mean,
                                    __bf16* out, size_t n, size_t per, float scale) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4* s = reinterpret_cast<const float4*>(xs + 8 * i);
  const float4 a = s[0], b = s[1];
  bf16x8 r;
  r[0] = (__bf16)((a.x - mean[i / per]) * scale);
  r[1] = (__bf16)a.y;
  r[2] = (__bf16)a.z;
  r[3] = (__bf16)a.w;
  r[4] = (__bf16)b.x;
  r[5] = (__bf16)b.y;
  r[6] = (__bf16)b.z;
  r[7] = (__bf16)b.w;
  store8(out + 8 * i, r);
}

__device__ inline float capped_expm1(float v, float scale) {
  v *= scale;
  return expm1f(v > 20.0f ? 20.0f : v);
}
__device__ inline float signed_expm1(float v, float scale) {
  const float s = (float)((0.0f < v) - (v < 0.0f));
  return s * capped_expm1(fabsf(v), scale);
}

// the core of window k of y [k][tile][tile][8], decoded, into the maps
__global__ void window_output_kernel(const float* __restrict__ y, WindowJobs j, float* d,
                                     float* mx, float* my, int Y, int tile, float scale) {
  const int k = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
  const int lx = j.lx[k], ly = j.ly[k];
  if (c >= lx * ly) return;
  const int x = j.cx[k] + c / ly, yy = j.cy[k] + c % ly;
  const float4 v = *reinterpret_cast<const float4*>(
      y + 8 * (((size_t)k * tile + x - j.wx[k]) * tile + yy - j.wy[k]));
  const size_t o = (size_t)x * Y + yy;
  const float dd = capped_expm1(v.x, scale);
  d[o] = dd < 0.0f ? 0.0f : dd;
  mx[o] = signed_expm1(v.y, scale);
  my[o] = signed_expm1(v.z, scale);
}

__global__ void f32_to_bf16_kernel(const float* __restrict__ x, __bf16* y, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (__bf16)x[i];
}

__global__ void bf16_to_f32_kernel(const __bf16* __restrict__ x, float* y, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (float)x[i];
}

}  // namespace shy_nn

using namespace shy_nn;

namespace {
thread_local std::string g_nn_err;
int nn_fail(const std::string& m) {
  g_nn_err = m;
  return SHY_NN_ERR;
}
int nn_check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return nn_fail(std::string(what) + ": " + hipGetErrorString(e));
  return 0;
}
inline unsigned blocks(size_t n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

// Compute units of the current device (looked up once per device).
int device_cus() {
  static std::atomic<int> cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int c = cus[dev].load(std::memory_order_relaxed);
  if (c == 0) {
    if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c < 1)
      c = 256;
    cus[dev].store(c, std::memory_order_relaxed);
  }
  return c;
}

// Persistent tile loop (conv_tiles_kernel): three blocks per compute unit
// over the layer's tiles of 16 x 16 pixels, 32 output channels per block.  A
// 64-channel layer takes two such blocks per tile: at 16 x 128^2, 32->64
// 31.1 -> 27.8 us and 64->64 41.7 -> 40.7 us against one 64-channel block
// at two blocks per CU (the 64-channel block needs 255 VGPRs).
// blocks per 32 output channels that run at once
long long tile_blocks(const ConvArgs& a) {
  return std::max(1LL, (long long)kTileBlocksPerCU * device_cus() / (a.Cout / 32));
}

template <int NT>
int launch_tiles_of(const ConvArgs& a, hipStream_t s, const char* what) {
  constexpr int MT = 2;
  const long long tiles = (long long)a.N * ((a.H + 4 * NT - 1) / (4 * NT)) * ((a.W + kTW - 1) / kTW);
  if (tiles > INT32_MAX) return nn_fail(std::string(what) + ": too many tiles");
  const long long cap = tile_blocks(a);
  // One tile per block, dealt out as blocks end, where a wide layer's blocks
  // would take one or two each (from 160 channels on a tile is long beside its
  // first loads; us at batch 16, 32^2 512 -> 512 channels 86 / 78, 3 x 104 x 152 256 ->
  // 256 from two tensors 70.5 / 65.9)
  const bool one = a.Cin > 128 && tiles > cap && tiles < 2 * cap;
  const dim3 g((unsigned)(one ? tiles : std::min(tiles, cap)), (unsigned)(a.Cout / (16 * MT)));
  if (a.x2) {
    if (a.res) conv_tiles_kernel<MT, NT, true, false, false, kEpiRes><<<g, 256, 0, s>>>(a);
    else conv_tiles_kernel<MT, NT, true, false, false, kEpiPlain><<<g, 256, 0, s>>>(a);
  } else if (a.head_w) {
    if (a.res) conv_tiles_kernel<MT, NT, false, true, false, kEpiRes><<<g, 256, 0, s>>>(a);
    else conv_tiles_kernel<MT, NT, false, true, false, kEpiPlain><<<g, 256, 0, s>>>(a);
  } else if (a.pool_y) {
    if (a.res) conv_tiles_kernel<MT, NT, false, false, true, kEpiRes><<<g, 256, 0, s>>>(a);
    else conv_tiles_kernel<MT, NT, false, false, true, kEpiPlain><<<g, 256, 0, s>>>(a);
  } else if (a.gres) {
    conv_tiles_kernel<MT, NT, false, false, false, kEpiGrad><<<g, 256, 0, s>>>(a);
  } else if (a.mask) {
    conv_tiles_kernel<MT, NT, false, false, false, kEpiMask><<<g, 256, 0, s>>>(a);
  } else {
    if (a.res) conv_tiles_kernel<MT, NT, false, false, false, kEpiRes><<<g, 256, 0, s>>>(a);
    else conv_tiles_kernel<MT, NT, false, false, false, kEpiPlain><<<g, 256, 0, s>>>(a);
  }
  return nn_check(what);
}

// 16 x 8 tiles where all of them run at once (twice the blocks, each half as
// long), or where 16 x 16 ones would be as many (maps of 8 rows and fewer).  Us
// with 16 x 8 / 16 x 16 tiles: 60 x 36 at batch 7 128 -> 128 channels 13.1 / 14.8, all
// 16 x 8 ones at once; not all of them: 48 x 80 at batch 10 96 -> 96 18.4 / 12.6, 224 ->
// 96 35.3 / 23.4, 88 x 24 at batch 9 128 -> 128 17.7 / 14.0.
int launch_tiles(const ConvArgs& a, hipStream_t s, const char* what) {
  const long long across = (long long)a.N * ((a.W + kTW - 1) / kTW);
  const long long tiles8 = across * ((a.H + 7) / 8), tiles16 = across * ((a.H + 15) / 16);
  return tiles8 <= tile_blocks(a) || tiles8 == tiles16 ? launch_tiles_of<2>(a, s, what)
                                                       : launch_tiles_of<4>(a, s, what);
}

// Cin and Cout multiples of 32: the tile loop for 3x3 (against one tile per
// block at batch 16: 32->32 at 256^2 50.7 -> 43.4 us, [up2, skip] 96->32 at 256^2
// 105 -> 83 us before its buffer accesses); conv_pf_kernel, 32 output channels
// per block (64-channel blocks ran 4-16% slower: half the blocks, and 210-256
// VGPRs), for 1x1 and for rows beyond the tile loop's offsets, with 16x16 tiles
// when they give >= 1024 blocks, else 16x8.
int launch_pf(const ConvArgs& a, int taps, hipStream_t s, const char* what) {
  if (taps == 9 && tile_rows_fit(a)) return launch_tiles(a, s, what);
  const long long tiles16 = (long long)a.N * ((a.H + 15) / 16) * ((a.W + kTW - 1) / kTW);
  const unsigned gy = (unsigned)(a.Cout / 32);
  const long long tiles8 = (long long)a.N * ((a.H + 7) / 8) * ((a.W + kTW - 1) / kTW);
  if (tiles8 > INT32_MAX) return nn_fail(std::string(what) + ": too many tiles");
  const bool big = taps == 9 || tiles16 * gy >= 1024;
  const dim3 g((unsigned)(big ? tiles16 : tiles8), gy);
  if (a.x2) conv_pf_kernel<9, 2, 4, true><<<g, 256, 0, s>>>(a);  // the input is [up2(x), x2]
  else if (a.head_w) conv_pf_kernel<9, 2, 4, false, true><<<g, 256, 0, s>>>(a);
  else if (taps == 9) conv_pf_kernel<9, 2, 4><<<g, 256, 0, s>>>(a);
  else if (big) conv_pf_kernel<1, 2, 4><<<g, 256, 0, s>>>(a);
  else conv_pf_kernel<1, 2, 2><<<g, 256, 0, s>>>(a);
  return nn_check(what);
}

// Device address of `scratch` on the current device: looked up once per
// device (on that device's first allocation-free call) and kept.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_dev[kMaxDevices] = {};

int noalloc_scratch(float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return nn_fail(std::string("noalloc: hipGetDevice: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return nn_fail("noalloc: device index beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return nn_fail(std::string("noalloc: hipGetSymbolAddress(scratch): ") +
                     hipGetErrorString(e));
    g_scratch_dev[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_dev[dev];
  return 0;
}
}  // namespace

extern "C" {

const char* shy_nn_last_error(void) { return g_nn_err.c_str(); }

int shy_nn_conv_fwd(const void* x, const void* w, const float* bias, const void* res, void* y_bf16,
                    float* y_f32, int N, int H, int W, int Cin, int Cout, int taps, int relu,
                    void* stream) {
  if (!x || !w || (!y_bf16 && !y_f32) || (y_bf16 && y_f32)) return nn_fail("conv_fwd: bad pointers");
  if ((uintptr_t)bias & 15) return nn_fail("conv_fwd: bias must be 16-byte aligned");
  if (N < 1 || H < 1 || W < 1 || Cin < 8 || Cin % 8 || Cout < 1 || (taps != 9 && taps != 1))
    return nn_fail("conv_fwd: need Cin a multiple of 8 and taps 9 or 1");
  ConvArgs a;
  a.x = (const __bf16*)x;
  a.w = (const __bf16*)w;
  a.bias = bias;
  a.res = (const __bf16*)res;
  a.y_bf = (__bf16*)y_bf16;
  a.y_f = y_f32;
  a.N = N; a.H = H; a.W = W; a.Cin = Cin; a.Cout = Cout; a.K = taps * Cin;
  a.relu = relu;
  a.x2 = nullptr;
  a.C1 = 0;
  a.gres = nullptr;
  a.mask = nullptr;
  const long long P = (long long)N * H * W;
  if (P > INT32_MAX / 2) return nn_fail("conv_fwd: too many pixels");
  hipStream_t s = (hipStream_t)stream;
  if (Cin % 32 == 0 && Cout % 32 == 0) return launch_pf(a, taps, s, "conv_fwd");
  if (Cin == 8 && taps == 9 && Cout % 32 == 0) {  // the first layer
    const int mt = Cout % 64 == 0 ? 4 : 2;
    const long long tiles = (long long)N * ((H + 15) / 16) * ((W + kTW - 1) / kTW);
    if (tiles > INT32_MAX) return nn_fail("conv_fwd: too many tiles");
    const dim3 g((unsigned)tiles, (unsigned)(Cout / (16 * mt)));
    if (mt == 4) conv_c8_kernel<4, 4><<<g, 256, 0, s>>>(a);
    else conv_c8_kernel<2, 4><<<g, 256, 0, s>>>(a);
    return nn_check("conv_fwd");
  }
  const unsigned gx = (unsigned)((P + 127) / 128);
  if (Cout > 16) {
    dim3 g(gx, (unsigned)((Cout + 31) / 32));
    if (taps == 9) conv_fwd_kernel<9, 2><<<g, 256, 0, s>>>(a);
    else conv_fwd_kernel<1, 2><<<g, 256, 0, s>>>(a);
  } else {
    dim3 g(gx, 1);
    if (taps == 9) conv_fwd_kernel<9, 1><<<g, 256, 0, s>>>(a);
    else conv_fwd_kernel<1, 1><<<g, 256, 0, s>>>(a);
  }
  return nn_check("conv_fwd");
}

int shy_nn_conv_fwd_head(const void* x, const void* w, const float* bias, const void* res,
                         void* y_bf16, const void* head_w, const float* head_b, float* head_y,
                         int N, int H, int W, int Cin, int head_c, int relu, void* stream) {
  if (!x || !w || !head_w || !head_y) return nn_fail("conv_fwd_head: bad pointers");
  if (((uintptr_t)bias | (uintptr_t)head_b | (uintptr_t)head_w) & 15)
    return nn_fail("conv_fwd_head: bias, head_w and head_b must be 16-byte aligned");
  if (N < 1 || H < 1 || W < 1 || (Cin != 32 && Cin != 64) || head_c < 4 || head_c > 16 ||
      head_c % 4)
    return nn_fail("conv_fwd_head: need Cin 32 or 64 and head_c in {4, 8, 12, 16}");
  if ((long long)N * H * W > INT32_MAX / 2) return nn_fail("conv_fwd_head: too many pixels");
  ConvArgs a;
  a.x = (const __bf16*)x;
  a.w = (const __bf16*)w;
  a.bias = bias;
  a.res = (const __bf16*)res;
  a.y_bf = (__bf16*)y_bf16;
  a.y_f = nullptr;
  a.N = N; a.H = H; a.W = W; a.Cin = Cin; a.Cout = 32; a.K = 9 * Cin;
  a.relu = relu;
  a.x2 = nullptr;
  a.C1 = 0;
  a.gres = nullptr;
  a.mask = nullptr;
  a.head_w = (const __bf16*)head_w;
  a.head_b = head_b;
  a.head_y = head_y;
  a.head_c = head_c;
  return launch_pf(a, 9, (hipStream_t)stream, "conv_fwd_head");
}

int shy_nn_conv_fwd_upcat(const void* x_half, const void* skip, const void* w, const float* bias,
                          const void* res, void* y_bf16, float* y_f32, int N, int H, int W,
                          int C1, int C2, int Cout, int relu, void* stream) {
  if (!x_half || !skip || !w || (!y_bf16 && !y_f32) || (y_bf16 && y_f32))
    return nn_fail("conv_fwd_upcat: bad pointers");
  if ((uintptr_t)bias & 15) return nn_fail("conv_fwd_upcat: bias must be 16-byte aligned");
  if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C1 < 32 || C1 % 32 || C2 < 32 || C2 % 32 ||
      Cout < 32 || Cout % 32)
    return nn_fail("conv_fwd_upcat: need even H, W and C1, C2, Cout multiples of 32");
  if ((long long)N * H * W > INT32_MAX / 2) return nn_fail("conv_fwd_upcat: too many pixels");
  ConvArgs a;
  a.x = (const __bf16*)x_half;
  a.x2 = (const __bf16*)skip;
  a.C1 = C1;
  a.w = (const __bf16*)w;
  a.bias = bias;
  a.res = (const __bf16*)res;
  a.y_bf = (__bf16*)y_bf16;
  a.y_f = y_f32;
  a.N = N; a.H = H; a.W = W; a.Cin = C1 + C2; a.Cout = Cout; a.K = 9 * (C1 + C2);
  a.relu = relu;
  a.gres = nullptr;
  a.mask = nullptr;
  return launch_pf(a, 9, (hipStream_t)stream, "conv_fwd_upcat");
}


int shy_nn_conv_fwd_pool(const void* x, const void* w, const float* bias, const void* res,
                         void* y_bf16, void* pool_y, int N, int H, int W, int Cin, int Cout,
                         int relu, void* stream) {
  if (!x || !w || !y_bf16 || !pool_y) return nn_fail("conv_fwd_pool: bad pointers");
  if (((uintptr_t)bias & 15) || ((uintptr_t)pool_y & 7))
    return nn_fail("conv_fwd_pool: bias must be 16-byte and pool_y 8-byte aligned");
  if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || Cin < 32 || Cin % 32 || Cout < 32 || Cout % 32)
    return nn_fail("conv_fwd_pool: need H, W even and Cin, Cout multiples of 32");
  if ((long long)N * H * W > INT32_MAX / 2) return nn_fail("conv_fwd_pool: too many pixels");
  ConvArgs a;
  a.W = W; a.Cin = Cin; a.Cout = Cout;
  if (!tile_rows_fit(a)) {
    // rows the tile loop does not take: the convolution, then the pool
    if (int r = shy_nn_conv_fwd(x, w, bias, res, y_bf16, nullptr, N, H, W, Cin, Cout, 9, relu,
                                stream))
      return r;
    return shy_nn_pool2(y_bf16, pool_y, N, H, W, Cout, 0, stream);
  }
  a.x = (const __bf16*)x;
  a.w = (const __bf16*)w;
  a.bias = bias;
  a.res = (const __bf16*)res;
  a.y_bf = (__bf16*)y_bf16;
  a.y_f = nullptr;
  a.N = N; a.H = H; a.W = W; a.Cin = Cin; a.Cout = Cout; a.K = 9 * Cin;
  a.relu = relu;
  a.x2 = nullptr;
  a.C1 = 0;
  a.gres = nullptr;
  a.mask = nullptr;
  a.pool_y = (__bf16*)pool_y;
  return launch_tiles(a, (hipStream_t)stream, "conv_fwd_pool");
}

// Work memory of shy_nn_unet_forward: per level three activations of its
// channels (stage output and two between), the pooled input of the next level.
static size_t unet_align(size_t bytes) { return (bytes + 255) / 256 * 256; }

// the levels' channels that the network's convolutions take: the fused head
// reads 32, the others are multiples of 32
static bool unet_channels(const int* ch) {
  for (int k = 0; k < 4; ++k)
    if (ch[k] < 32 || ch[k] % 32) return false;
  return ch[0] == 32;
}

long long shy_nn_unet_work_bytes(const int* ch, int N, int H, int W) {
  if (!ch || !unet_channels(ch) || N < 1 || H < 8 || W < 8 || H % 8 || W % 8) return -1;
  size_t sum = 0;
  for (int k = 0; k < 4; ++k) {
    const size_t p = (size_t)N * (H >> k) * (W >> k) * 2;
    sum += 3 * unet_align(p * ch[k]) + (k < 3 ? unet_align(p / 4 * ch[k]) : 0);
  }
  return (long long)sum;
}

int shy_nn_unet_forward(const void* x, const void* const* w, const float* const* b, const int* ch,
                        int cin, int head_c, void* work, long long work_bytes, float* out, int N,
                        int H, int W, void* stream) {
  if (!x || !w || !b || !ch || !work || !out) return nn_fail("unet_forward: bad pointers");
  // before the first launch
  if (!unet_channels(ch) || cin < 8 || cin % 8 || head_c < 4 || head_c > 16 || head_c % 4)
    return nn_fail("unet_forward: need ch[0] = 32, ch[1..3] multiples of 32, cin a multiple of 8, "
                   "head_c in {4, 8, 12, 16}");
  const long long need = shy_nn_unet_work_bytes(ch, N, H, W);
  if (need < 0) return nn_fail("unet_forward: H and W must be multiples of 8");
  if (work_bytes < need) return nn_fail("unet_forward: work memory too small");
  char* at = (char*)work;
  auto take = [&](size_t bytes) {
    void* p = at;
    at += unet_align(bytes);
    return p;
  };
  void *ya[4], *yb[4], *yc[4], *pool[3];
  for (int k = 0; k < 4; ++k) {
    const size_t p = (size_t)N * (H >> k) * (W >> k) * 2;
    ya[k] = take(p * ch[k]);
    yb[k] = take(p * ch[k]);
    yc[k] = take(p * ch[k]);
    if (k < 3) pool[k] = take(p / 4 * ch[k]);
  }
  int c = 0;  // convolution
  auto conv = [&](const void* in, void* y, const void* res, int k, int ci) {
    const int r = shy_nn_conv_fwd(in, w[c], b[c], res, y, nullptr, N, H >> k, W >> k, ci, ch[k], 9,
                                  1, stream);
    ++c;
    return r;
  };
  const void* h = x;
  for (int k = 0; k < 4; ++k) {
    if (int r = conv(h, ya[k], nullptr, k, k == 0 ? cin : ch[k - 1])) return r;
    if (int r = conv(ya[k], yb[k], nullptr, k, ch[k])) return r;
    if (k == 3) {
      if (int r = conv(yb[k], yc[k], ya[k], k, ch[k])) return r;
    } else {
      if (int r = shy_nn_conv_fwd_pool(yb[k], w[c], b[c], ya[k], yc[k], pool[k], N, H >> k, W >> k,
                                       ch[k], ch[k], 1, stream))
        return r;
      ++c;
      h = pool[k];
    }
  }
  // decoder stages take the encoder's ya, yb and, but for the last, write over
  // its skip after reading it
  for (int k = 2; k >= 0; --k) {
    // w and b list the decoder stages from level 0 on
    c = 12 + 3 * k;
    if (int r = shy_nn_conv_fwd_upcat(yc[k + 1], yc[k], w[c], b[c], nullptr, ya[k], nullptr, N,
                                      H >> k, W >> k, ch[k + 1], ch[k], ch[k], 1, stream))
      return r;
    ++c;
    if (int r = conv(ya[k], yb[k], nullptr, k, ch[k])) return r;
    if (k > 0) {
      if (int r = conv(yb[k], yc[k], ya[k], k, ch[k])) return r;
    } else if (int r = shy_nn_conv_fwd_head(yb[k], w[c], b[c], ya[k], nullptr, w[21], b[21], out, N,
                                            H, W, ch[0], head_c, 1, stream)) {
      return r;
    }
  }
  return 0;
}

int shy_nn_conv_dgrad(const void* g, const void* wf, const void* gres, const void* mask,
                      void* dx_bf16, int N, int H, int W, int Cin, int Cout, int taps,
                      void* stream) {
  if (!g || !wf || !dx_bf16) return nn_fail("conv_dgrad: bad pointers");
  if (N < 1 || H < 1 || W < 1 || Cin < 32 || Cin % 32 || Cout < 32 || Cout % 32 ||
      (taps != 9 && taps != 1))
    return nn_fail("conv_dgrad: need Cin and Cout multiples of 32 and taps 9 or 1");
  if ((long long)N * H * W > INT32_MAX / 2) return nn_fail("conv_dgrad: too many pixels");
  ConvArgs a;
  a.x = (const __bf16*)g;
  a.w = (const __bf16*)wf;
  a.bias = nullptr;
  a.res = nullptr;
  a.y_bf = (__bf16*)dx_bf16;
  a.y_f = nullptr;
  // the data gradient is the convolution of g (Cout channels) with the
  // flipped weights into Cin channels
  a.N = N; a.H = H; a.W = W; a.Cin = Cout; a.Cout = Cin; a.K = taps * Cout;
  a.relu = 0;
  a.x2 = nullptr;
  a.C1 = 0;
  a.gres = (const __bf16*)gres;
  a.mask = (const __bf16*)mask;
  return launch_pf(a, taps, (hipStream_t)stream, "conv_dgrad");
}

int shy_nn_flip_weights(const void* w, void* wf, int Cin, int Cout, int taps, void* stream) {
  if (!w || !wf || (taps != 9 && taps != 1)) return nn_fail("flip_weights: bad argument");
  const int n = Cin * Cout * taps;
  flip_weights_kernel<<<blocks(n), 256, 0, (hipStream_t)stream>>>((const __bf16*)w, (__bf16*)wf,
                                                                  Cin, Cout, taps);
  return nn_check("flip_weights");
}

inline bool a16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// pixels per partial of shy_nn_bias_grad: at least 2048 (two 1024-thread blocks
// per CU on the largest layers, eight rows in flight per thread)
static int bias_rows_per_block(int P, int part_rows) {
  return std::max((P + part_rows - 1) / part_rows, 2048);
}

// The weight gradient by wgrad_lds_kernel, of x or (C1 > 0) [up2(x), x2];
// part holds part_splits partials.  With db the bias gradient too, bias_part
// holding bias_rows partials.
static int wgrad_lds(const void* x, const void* x2, int C1, const void* g, float* dw, float* part,
                     int part_splits, float* db, float* bias_part, int bias_rows, int N, int H,
                     int W, int Cin, int Cout, hipStream_t s) {
  WgArgs b;
  b.x = (const __bf16*)x;
  b.x2 = (const __bf16*)x2;
  b.C1 = C1;
  b.g = (const __bf16*)g;
  b.part = part;
  b.N = N; b.H = H; b.W = W; b.Cin = Cin; b.Cout = Cout; b.K = 9 * Cin;
  b.tiles_x = (W + kWgTW - 1) / kWgTW;
  b.tiles_y = (H + kWgTH - 1) / kWgTH;
  const long long tiles = (long long)N * b.tiles_x * b.tiles_y;
  if (tiles > INT32_MAX) return nn_fail("conv_wgrad: too many tiles");
  b.tiles = (int)tiles;
  const int bxy = (Cout / 32) * (Cin / 32);
  // about 1024 blocks, at most part_splits partials, at least one tile each;
  // the ranges of tiles are part of the order of the sums (wgrad_lds_kernel)
  long long splits = std::max(1LL, std::min<long long>((1024 + bxy - 1) / bxy, tiles));
  splits = std::min<long long>(splits, part_splits);
  b.tiles_per_split = (int)((tiles + splits - 1) / splits);
  splits = (tiles + b.tiles_per_split - 1) / b.tiles_per_split;
  // a range of tiles per XCD where the 8 XCDs then have equal work to 1/8.  Ranges
  // on their XCD / channel blocks dealt out, us at batch 16: 2 ranges, 32^2 512 ->
  // 512 channels 447 / 135; 4, 16^2 1024 -> 1024 at batch 2 220 / 113; 10, 64^2
  // 224 -> 224 171 / 106; 26, 32^2 128 -> 128 23.0 / 20.0; 29, 64^2 128 -> 128 41.1 /
  // 49.5; 46, 128^2 160 -> 64 83.0 / 112
  b.xcds = (splits + 7) / 8 * 64 <= splits * 9 ? 8 : 1;
  b.blocks = (int)((splits + b.xcds - 1) / b.xcds * b.xcds * bxy);
  b.bias_part = bias_part;
  b.bias_rows = 0;
  int nb = 0;
  if (db) {
    const int P = N * H * W;
    b.bias_rows = bias_rows_per_block(P, bias_rows);
    nb = (P + b.bias_rows - 1) / b.bias_rows;
  }
  wgrad_lds_kernel<<<(unsigned)(b.blocks + nb * (Cout / 32)), kWgThreads, 0, s>>>(b);
  if (int r = nn_check("conv_wgrad")) return r;
  const int n = Cout * b.K;
  wgrad_reduce_kernel<<<(n + 31) / 32 + (db ? Cout / 8 : 0), 256, 0, s>>>(
      part, dw, n, (int)splits, bias_part, db, Cout, nb);
  return nn_check("wgrad_reduce");
}

int shy_nn_conv_wgrad(const void* x, const void* g, float* dw, float* part, int part_splits,
                      int N, int H, int W, int Cin, int Cout, int taps, void* stream) {
  if (!x || !g || !dw || !part || part_splits < 1) return nn_fail("conv_wgrad: bad pointers");
  if (Cin % 8 || Cout % 8 || (taps != 9 && taps != 1)) return nn_fail("conv_wgrad: channels must be multiples of 8");
  const long long P = (long long)N * H * W;
  if (taps == 9 && Cin % 32 == 0 && Cout % 32 == 0)
    return wgrad_lds(x, nullptr, 0, g, dw, part, part_splits, nullptr, nullptr, 0, N, H, W, Cin,
                     Cout, (hipStream_t)stream);
  int chunk = (int)((P + part_splits - 1) / part_splits);

  chunk = (chunk + 31) / 32 * 32;
  const int splits = (int)((P + chunk - 1) / chunk);
  WgradArgs a;
  a.x = (const __bf16*)x;
  a.g = (const __bf16*)g;
  a.part = part;
  a.N = N; a.H = H; a.W = W; a.Cin = Cin; a.Cout = Cout; a.K = taps * Cin; a.taps = taps;
  a.chunk = chunk;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((unsigned)((Cout + 31) / 32), (unsigned)((a.K + 31) / 32), (unsigned)splits);
  conv_wgrad_kernel<<<grid, 64, 0, s>>>(a);
  if (int r = nn_check("conv_wgrad")) return r;
  const int n = Cout * a.K;
  wgrad_reduce_kernel<<<(n + 31) / 32, 256, 0, s>>>(part, dw, n, splits, nullptr, nullptr, 0, 0);
  return nn_check("wgrad_reduce");
}

int shy_nn_conv_wgrad_noalloc(const void* x, const void* g, float* dw, int N, int H, int W,
                              int Cin, int Cout, int taps, void* stream) {
  if (Cin < 1 || Cout < 1 || (taps != 9 && taps != 1))
    return nn_fail("conv_wgrad_noalloc: bad shape");
  const size_t per = (size_t)Cout * taps * Cin;
  if (per > (size_t)SHY_NN_NOALLOC_FLOATS)
    return nn_fail("conv_wgrad_noalloc: Cout*taps*Cin = " + std::to_string(per) +
                   " floats exceeds the scratch of " + std::to_string(SHY_NN_NOALLOC_FLOATS));
  float* part = nullptr;
  if (int r = noalloc_scratch(&part)) return r;
  const int splits = (int)std::min<size_t>((size_t)SHY_NN_NOALLOC_FLOATS / per,
                                           (size_t)SHY_NN_NOALLOC_MAX_SPLITS);
  return shy_nn_conv_wgrad(x, g, dw, part, splits, N, H, W, Cin, Cout, taps, stream);
}

int shy_nn_bias_grad(const void* g, float* db, float* part, int part_rows, int P, int C,
                     void* stream) {
  if (!g || !db || !part || C < 1 || C > 1024 || P < 1 || part_rows < 1)
    return nn_fail("bias_grad: bad argument");
  hipStream_t s = (hipStream_t)stream;
  if (C % 8 == 0 && ((uintptr_t)g & 15) == 0 && ((uintptr_t)part & 15) == 0) {
    const int rows = bias_rows_per_block(P, part_rows);
    const int nb = (P + rows - 1) / rows;
    bias_grad_v8_kernel<<<nb, 1024, 0, s>>>((const __bf16*)g, part, P, C, rows);
    if (int r = nn_check("bias_grad")) return r;
    bias_reduce_kernel<<<1, 1024, 0, s>>>(part, db, C, nb);
    return nn_check("bias_grad_reduce");
  }
  const int rows = (P + part_rows - 1) / part_rows;
  const int nb = (P + rows - 1) / rows;
  bias_grad_kernel<<<nb, 256, 0, s>>>((const __bf16*)g, part, P, C, rows);
  if (int r = nn_check("bias_grad")) return r;
  wgrad_reduce_kernel<<<(C + 31) / 32, 256, 0, s>>>(part, db, C, nb, nullptr, nullptr, 0,
                                                     0);
  return nn_check("bias_grad_reduce");
}

int shy_nn_conv_wgrad_bias(const void* x, const void* g, float* dw, float* db, float* part,
                           int part_splits, float* bias_part, int bias_rows, int N, int H, int W,
                           int Cin, int Cout, int taps, void* stream) {
  // the tiled weight gradient's launches take the bias sums along, where these
  // are shy_nn_bias_grad's 8-channel ones
  const long long P = (long long)N * H * W;
  if (x && g && dw && db && part && part_splits > 0 && bias_part && bias_rows > 0 && taps == 9 &&
      Cin > 0 && Cout > 0 && Cout <= 1024 && Cin % 32 == 0 && Cout % 32 == 0 && P > 0 &&
      P <= INT32_MAX && a16(g) && a16(bias_part))
    return wgrad_lds(x, nullptr, 0, g, dw, part, part_splits, db, bias_part, bias_rows, N, H, W,
                     Cin, Cout, (hipStream_t)stream);
  if (int r = shy_nn_conv_wgrad(x, g, dw, part, part_splits, N, H, W, Cin, Cout, taps, stream))
    return r;
  return shy_nn_bias_grad(g, db, bias_part, bias_rows, N * H * W, Cout, stream);
}

int shy_nn_conv_wgrad_bias_cat(const void* x_half, const void* skip, const void* g, float* dw,
                               float* db, float* part, int part_splits, float* bias_part,
                               int bias_rows, int N, int H, int W, int C1, int C2, int Cout,
                               void* stream) {
  if (!x_half || !skip || !g || !dw || !db || !part || part_splits < 1 || !bias_part ||
      bias_rows < 1)
    return nn_fail("conv_wgrad_bias_cat: bad pointers");
  if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C1 < 32 || C1 % 32 || C2 < 32 || C2 % 32 ||
      Cout < 32 || Cout % 32 || Cout > 1024 || (long long)N * H * W > INT32_MAX)
    return nn_fail("conv_wgrad_bias_cat: need H, W even and C1, C2, Cout multiples of 32");
  if (!a16(g) || !a16(bias_part)) {  // shy_nn_bias_grad's element-wise sums
    if (int r = shy_nn_bias_grad(g, db, bias_part, bias_rows, N * H * W, Cout, stream)) return r;
    db = nullptr;
  }
  return wgrad_lds(x_half, skip, C1, g, dw, part, part_splits, db, bias_part, bias_rows, N, H, W,
                   C1 + C2, Cout, (hipStream_t)stream);
}

int shy_nn_conv_wgrad_bias_upcat(const void* x_half, const void* skip, const void* g, float* dw,
                                 float* db, float* part, int part_splits, int N, int H, int W,
                                 int C1, int C2, int Cout, void* stream) {
  if (!x_half || !skip || !g || !dw || !db || !part || part_splits < 1)
    return nn_fail("conv_wgrad_bias_upcat: bad pointers");
  if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C1 < 32 || C1 % 32 || C2 < 32 || C2 % 32 ||
      Cout < 32 || Cout % 32 || Cout > 1024 || (long long)N * H * W > INT32_MAX)
    return nn_fail("conv_wgrad_bias_upcat: need H, W even and C1, C2, Cout multiples of 32");
  // the bias partials first, in the memory of the others (at least 576 Cout
  // floats)
  const size_t rows = std::min<size_t>(1024, (size_t)part_splits * 9 * (C1 + C2));
  if (int r = shy_nn_bias_grad(g, db, part, (int)rows, N * H * W, Cout, stream)) return r;
  return wgrad_lds(x_half, skip, C1, g, dw, part, part_splits, nullptr, nullptr, 0, N, H, W,
                   C1 + C2, Cout, (hipStream_t)stream);
}

int shy_nn_relu_bwd(const void* y, const void* g, void* out, size_t n, void* stream) {
  if (n % 8 == 0 && a16(y) && a16(g) && a16(out))
    relu_bwd_v8_kernel<<<blocks(n / 8), 256, 0, (hipStream_t)stream>>>(
        (const __bf16*)y, (const __bf16*)g, (__bf16*)out, n / 8);
  else
    relu_bwd_kernel<<<blocks(n), 256, 0, (hipStream_t)stream>>>((const __bf16*)y,
                                                                 (const __bf16*)g, (__bf16*)out, n);
  return nn_check("relu_bwd");
}

int shy_nn_pool2(const void* x, void* y, int N, int H, int W, int C, int backward, void* stream) {
  if (H % 2 || W % 2) return nn_fail("pool2: H and W must be even");
  hipStream_t s = (hipStream_t)stream;
  const bool v8 = C % 8 == 0 && a16(x) && a16(y);
  if (v8 && !backward)
    pool2_fwd_v8_kernel<<<blocks((size_t)N * H * W * C / 32), 256, 0, s>>>(
        (const __bf16*)x, (__bf16*)y, N, H, W, C);
  else if (v8)
    pool2_bwd_v8_kernel<<<blocks((size_t)N * H * W * C / 8), 256, 0, s>>>(
        (const __bf16*)x, (__bf16*)y, N, H, W, C);
  else if (!backward)
    pool2_fwd_kernel<<<blocks((size_t)N * H * W * C / 4), 256, 0, s>>>((const __bf16*)x, (__bf16*)y,
                                                                       N, H, W, C);
  else
    pool2_bwd_kernel<<<blocks((size_t)N * H * W * C), 256, 0, s>>>((const __bf16*)x, (__bf16*)y, N,
                                                                   H, W, C);
  return nn_check("pool2");
}

int shy_nn_up2(const void* x, void* y, int N, int H, int W, int C, int Cy, int c_off, int backward,
               void* stream) {
  if (c_off < 0 || c_off + C > Cy) return nn_fail("up2: channel range outside the target");
  hipStream_t s = (hipStream_t)stream;
  const bool v8 = C % 8 == 0 && Cy % 8 == 0 && c_off % 8 == 0 && a16(x) && a16(y);
  if (v8 && !backward)
    up2_fwd_v8_kernel<<<blocks((size_t)N * 4 * H * W * C / 8), 256, 0, s>>>(
        (const __bf16*)x, (__bf16*)y, N, H, W, C, Cy, c_off);
  else if (v8)
    up2_bwd_v8_kernel<<<blocks((size_t)N * H * W * C / 8), 256, 0, s>>>(
        (const __bf16*)x, (__bf16*)y, nullptr, N, H, W, C, Cy, c_off);
  else if (!backward)
    up2_fwd_kernel<<<blocks((size_t)N * 4 * H * W * C), 256, 0, s>>>(
        (const __bf16*)x, (__bf16*)y, N, H, W, C, Cy, c_off);
  else
    up2_bwd_kernel<<<blocks((size_t)N * H * W * C), 256, 0, s>>>((const __bf16*)x, (__bf16*)y, N, H,
                                                                 W, C, Cy, c_off);
  return nn_check("up2");
}

int shy_nn_up2_bwd_relu(const void* gy, const void* y, void* gx, int N, int H, int W, int C, int Cy,
                        int c_off, void* stream) {
  if (!gy || !y || !gx) return nn_fail("up2_bwd_relu: bad pointers");
  if (N < 1 || H < 1 || W < 1 || C < 8 || C % 8 || Cy % 8 || c_off % 8 || c_off < 0 ||
      c_off + C > Cy || !a16(gy) || !a16(y) || !a16(gx))
    return nn_fail("up2_bwd_relu: need channels in multiples of 8, inside the target, 16-byte "
                   "aligned tensors");
  up2_bwd_v8_kernel<<<blocks((size_t)N * H * W * C / 8), 256, 0, (hipStream_t)stream>>>(
      (const __bf16*)gy, (__bf16*)gx, (const __bf16*)y, N, H, W, C, Cy, c_off);
  return nn_check("up2_bwd_relu");
}

int shy_nn_skip_bwd(const void* gp, const void* gu, const void* y, void* out, int N, int H, int W,
                    int C, int Cu, int c_off, void* stream) {
  if (!gp || !gu || !y || !out) return nn_fail("skip_bwd: bad pointers");
  if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C < 8 || C % 8 || Cu % 8 || c_off % 8 ||
      c_off < 0 || c_off + C > Cu || !a16(gp) || !a16(gu) || !a16(y) || !a16(out))
    return nn_fail("skip_bwd: need H, W even, channels in multiples of 8, inside the source, "
                   "16-byte aligned tensors");
  skip_bwd_v8_kernel<<<blocks((size_t)N * H * W * C / 8), 256, 0, (hipStream_t)stream>>>(
      (const __bf16*)gp, (const __bf16*)gu, (const __bf16*)y, (__bf16*)out, N, H, W, C, Cu, c_off);
  return nn_check("skip_bwd");
}

int shy_nn_channels(const void* src, void* dst, size_t P, int C, int Cy, int c_off, int dir,
                    void* stream) {
  if (c_off < 0 || c_off + C > Cy) return nn_fail("channels: range outside the target");
  if (C % 8 == 0 && Cy % 8 == 0 && c_off % 8 == 0 && a16(src) && a16(dst))
    channels_copy_v8_kernel<<<blocks(P * C / 8), 256, 0, (hipStream_t)stream>>>(
        (const __bf16*)src, (__bf16*)dst, P, C, Cy, c_off, dir);
  else
    channels_copy_kernel<<<blocks(P * C), 256, 0, (hipStream_t)stream>>>(
        (const __bf16*)src, (__bf16*)dst, P, C, Cy, c_off, dir);
  return nn_check("channels");
}

int shy_nn_add(const void* a, const void* b, void* y, size_t n, void* stream) {
  if (n % 8 == 0 && a16(a) && a16(b) && a16(y))
    add_v8_kernel<<<blocks(n / 8), 256, 0, (hipStream_t)stream>>>(
        (const __bf16*)a, (const __bf16*)b, (__bf16*)y, n / 8);
  else
    add_kernel<<<blocks(n), 256, 0, (hipStream_t)stream>>>((const __bf16*)a, (const __bf16*)b,
                                                            (__bf16*)y, n);
  return nn_check("add");
}

int shy_nn_mse(const float* y, const float* t, const float* mask, void* g_bf16, float* part,
               size_t n, float inv_count, void* stream) {
  mse_kernel<<<blocks(n), 256, 0, (hipStream_t)stream>>>(y, t, mask, (__bf16*)g_bf16, part, n,
                                                          inv_count);
  return nn_check("mse");
}

int shy_nn_adam(float* w, const float* g, float* m, float* v, void* w_bf16, size_t n, float lr,
                float b1, float b2, float eps, int step, float weight_decay, void* stream) {
  if (step < 1) return nn_fail("adam: step must be >= 1");
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  const AdamStep a{lr, b1, b2, eps, c1, c2, weight_decay};
  adam_kernel<<<blocks(n), 256, 0, (hipStream_t)stream>>>(a, w, g, m, v, (__bf16*)w_bf16, n);
  return nn_check("adam");
}

int shy_nn_adam_conv_bias(float* w, const float* g, float* m, float* v, void* w_bf16,
                          void* wf_bf16, int Cin, int Cout, int taps, float* b, const float* bg,
                          float* bm, float* bv, float lr, float b1, float b2, float eps, int step,
                          float weight_decay, void* stream) {
  if (step < 1) return nn_fail("adam_conv: step must be >= 1");
  if (!w || !g || !m || !v || !w_bf16 || !wf_bf16 || Cin < 1 || Cout < 1 ||
      (taps != 9 && taps != 1) || (b && (!bg || !bm || !bv)))
    return nn_fail("adam_conv: bad argument");
  const size_t n = (size_t)Cout * taps * Cin;
  const int nb = b ? Cout : 0;
  if (n > (size_t)INT32_MAX) return nn_fail("adam_conv: too many weights");
  const AdamStep a{lr, b1, b2, eps, 1.0f - powf(b1, (float)step), 1.0f - powf(b2, (float)step),
                   weight_decay};
  adam_conv_kernel<<<blocks(n + nb), 256, 0, (hipStream_t)stream>>>(
      a, w, g, m, v, (__bf16*)w_bf16, (__bf16*)wf_bf16, Cin, Cout, taps, b, bg, bm, bv, nb);
  return nn_check("adam_conv");
}

int shy_nn_adam_conv(float* w, const float* g, float* m, float* v, void* w_bf16, void* wf_bf16,
                     int Cin, int Cout, int taps, float lr, float b1, float b2, float eps, int step,
                     float weight_decay, void* stream) {
  return shy_nn_adam_conv_bias(w, g, m, v, w_bf16, wf_bf16, Cin, Cout, taps, nullptr, nullptr,
                               nullptr, nullptr, lr, b1, b2, eps, step, weight_decay, stream);
}

int shy_nn_flow_features(const float* h, const float* d, const float* mx, const float* my,
                         const long long* strides, float* feats, int X, int Y, float slope,
                         float scale, void* stream) {
  if (!h || !d || !mx || !my || !strides || !feats || X < 1 || Y < 1 || !a16(feats))
    return nn_fail("flow_features: bad argument");
  const FlowMaps m{{h, strides[0], strides[1]}, {d, strides[2], strides[3]},
                   {mx, strides[4], strides[5]}, {my, strides[6], strides[7]}};
  flow_features_kernel<<<blocks((size_t)X * Y), 256, 0, (hipStream_t)stream>>>(m, feats, X, Y, slope,
                                                                               scale);
  return nn_check("flow_features");
}

// jobs: {wx, cx, lx, wy, cy, ly} per window; each must lie in the map
static int window_jobs(const int* jobs, int n, int X, int Y, int tile, WindowJobs& w) {
  if (!jobs || n < 1 || n > kJobs || tile < 1 || tile > 32767)
    return nn_fail("windows: need 1 to 32 windows");
  for (int k = 0; k < n; ++k) {
    const int* j = jobs + 6 * k;
    w.wx[k] = j[0]; w.cx[k] = j[1]; w.lx[k] = j[2];
    w.wy[k] = j[3]; w.cy[k] = j[4]; w.ly[k] = j[5];
    if (j[0] < 0 || j[0] > X - tile || j[3] < 0 || j[3] > Y - tile || j[2] < 1 || j[5] < 1 ||
        j[1] < j[0] || j[1] - j[0] > tile - j[2] || j[4] < j[3] || j[4] - j[3] > tile - j[5])
      return nn_fail("windows: a window outside the map, or its core outside it");
  }
  return 0;
}

int shy_nn_window_copy(const float* feats, const int* jobs, int n, float* out, int X, int Y,
                       int tile, void* stream) {
  WindowJobs w{};
  if (!feats || !out || !a16(feats) || !a16(out)) return nn_fail("window_copy: bad pointers");
  if (int r = window_jobs(jobs, n, X, Y, tile, w)) return r;
  window_copy_kernel<<<dim3(blocks((size_t)tile * tile * 2), (unsigned)n), 256, 0,
                       (hipStream_t)stream>>>(feats, out, w, Y, tile);
  return nn_check("window_copy");
}

int shy_nn_window_input(const float* xs, const float* mean, void* out, int n, int tile, float scale,
                        void* stream) {
  if (!xs || !mean || !out || n < 1 || tile < 1 || !a16(xs) || !a16(out))
    return nn_fail("window_input: bad argument");
  const size_t per = (size_t)tile * tile;
  window_input_kernel<<<blocks(per * n), 256, 0, (hipStream_t)stream>>>(xs, mean, (__bf16*)out,
                                                                        per * n, per, scale);
  return nn_check("window_input");
}

int shy_nn_window_output(const float* y, const int* jobs, int n, float* d, float* mx, float* my,
                         int X, int Y, int tile, float scale, void* stream) {
  WindowJobs w{};
  if (!y || !d || !mx || !my || !a16(y)) return nn_fail("window_output: bad pointers");
  if (int r = window_jobs(jobs, n, X, Y, tile, w)) return r;
  int most = 0;
  for (int k = 0; k < n; ++k) most = std::max(most, w.lx[k] * w.ly[k]);
  window_output_kernel<<<dim3(blocks((size_t)most), (unsigned)n), 256, 0, (hipStream_t)stream>>>(
      y, w, d, mx, my, Y, tile, scale);
  return nn_check("window_output");
}

int shy_nn_cast(const void* src, void* dst, size_t n, int to_bf16, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (to_bf16)
    f32_to_bf16_kernel<<<blocks(n), 256, 0, s>>>((const float*)src, (__bf16*)dst, n);
  else
    bf16_to_f32_kernel<<<blocks(n), 256, 0, s>>>((const __bf16*)src, (float*)dst, n);
  return nn_check("cast");
}

}  // extern "C"
