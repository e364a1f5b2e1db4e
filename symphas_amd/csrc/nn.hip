// nn.hip - BF16 MFMA convolution kernels of the learned surrogate
// (include/sps_nn.h).
//
// Forward (and backward-data, which is the forward kernel with flipped,
// transposed weights) is an implicit GEMM: M = output channels, N = pixels,
// K = 9 taps x input channels, on v_mfma_f32_16x16x32_bf16.  Operand layout
// of that instruction on gfx950 (wave64):
//   A (16 x 32, M x K): lane l holds A[l % 16][8*(l/16) + 0..7]
//   B (32 x 16, K x N): lane l holds B[8*(l/16) + 0..7][l % 16]
//   D (16 x 16):        lane l holds D[4*(l/16) + 0..3][l % 16]
// With NHWC activations and [tap][out][in] weights both A (weights) and B
// (pixels) fragments are single 16-byte loads, so the kernel streams straight
// from L1/L2; each wave owns 16*NT output channels x 64 pixels, reuses every
// weight fragment 4 times and every pixel fragment NT times, and stores 4
// consecutive output channels of a pixel per lane (8 bytes).
//
// The weight gradient reduces over pixels, which are strided in NHWC, so it
// stages a block of pixels of dpre and of the input with its halo in LDS and
// reads the fragments from there transposed (ds_read_b64_tr_b16).
#include <algorithm>
#include <cstdint>
#include <initializer_list>

#include "common.hpp"
#include "lanes.hpp"
#include "../../include/sps_nn.h"

namespace sps {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even: gfx950's v_cvt_pk_bf16_f32 (a NaN
// stays a quiet NaN).  pack_bf16 converts two values in one instruction.
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint16_t f2bf(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{lo, hi}, bf16x2v));
}
__device__ __forceinline__ float bf2f(uint16_t h) {
  return __uint_as_float((uint32_t)h << 16);
}

// v * sigmoid(v) with the hardware reciprocal (1 ulp; the result is rounded
// to BF16 or feeds BF16 data)
__device__ __forceinline__ float silu(float v) {
  return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
}

__device__ __forceinline__ bf16x8 load_frag(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(p));
}

// 4 consecutive BF16 values as one 8-byte access (callers keep 8-byte
// alignment: channel offsets are multiples of 4)
__device__ __forceinline__ void store4(uint16_t* p, const float (&v)[4]) {
  const uint32_t lo = pack_bf16(v[0], v[1]);
  const uint32_t hi = pack_bf16(v[2], v[3]);
  *reinterpret_cast<uint2*>(p) = make_uint2(lo, hi);
}
__device__ __forceinline__ void load4(const uint16_t* p, float (&v)[4]) {
  const uint2 q = *reinterpret_cast<const uint2*>(p);
  v[0] = bf2f((uint16_t)(q.x & 0xffffu));
  v[1] = bf2f((uint16_t)(q.x >> 16));
  v[2] = bf2f((uint16_t)(q.y & 0xffffu));
  v[3] = bf2f((uint16_t)(q.y >> 16));
}
// 8 consecutive BF16 values as one 16-byte access (16-byte aligned)
__device__ __forceinline__ void store8(uint16_t* p, const float (&v)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
  *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}
__device__ __forceinline__ void load8(const uint16_t* p, float (&v)[8]) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = bf2f((uint16_t)(w[i] & 0xffffu));
    v[2 * i + 1] = bf2f((uint16_t)(w[i] >> 16));
  }
}

__device__ __forceinline__ int wrapi(int v, int n) {
  return v < 0 ? v + n : (v >= n ? v - n : v);
}

template <int NT, int EPI>
__global__ __launch_bounds__(256) void conv_fwd(
    const uint16_t* __restrict__ x, int N, int H, int W, int C,
    const uint16_t* __restrict__ wt, const float* __restrict__ bias, int K,
    int act, const uint16_t* __restrict__ skip, uint16_t* __restrict__ y,
    uint16_t* __restrict__ pre, int npix) {
  // D = W (out channels x in channels) * X (in channels x pixels): rows of D
  // are output channels, so lane l ends with 4 consecutive channels of one
  // pixel and stores them as one 8-byte word.
  const int lane = threadIdx.x & 63;
  const int p0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 64;
  if (p0 >= npix) return;
  const int k0 = blockIdx.y * 16 * NT;
  const int HW = H * W;
  const int cq = (lane >> 4) * 8;
  int pn[4], ph[4], pw[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int p = p0 + 16 * m + (lane & 15);
    pn[m] = p / HW;
    const int r = p - pn[m] * HW;
    ph[m] = r / W;
    pw[m] = r - ph[m] * W;
  }
  f32x4v acc[NT][4];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[j][m] = f32x4v{0.f, 0.f, 0.f, 0.f};

  for (int tap = 0; tap < 9; ++tap) {
    const int dr = tap / 3 - 1, ds = tap % 3 - 1;
    const uint16_t* xrow[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int hh = wrapi(ph[m] + dr, H), ww = wrapi(pw[m] + ds, W);
      xrow[m] = x + ((int64_t)(pn[m] * H + hh) * W + ww) * C + cq;
    }
    const uint16_t* wrow = wt + ((int64_t)tap * K + k0 + (lane & 15)) * C + cq;
#pragma unroll 2
    for (int c0 = 0; c0 < C; c0 += 32) {
      bf16x8 a[NT], b[4];
#pragma unroll
      for (int j = 0; j < NT; ++j) a[j] = load_frag(wrow + (int64_t)j * 16 * C + c0);
#pragma unroll
      for (int m = 0; m < 4; ++m) b[m] = load_frag(xrow[m] + c0);
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          acc[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], b[m],
                                                              acc[j][m], 0, 0, 0);
    }
  }

#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int ch = k0 + 16 * j + 4 * (lane >> 4);  // 4 consecutive channels
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
      for (int i = 0; i < 4; ++i) bv[i] = bias[ch + i];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int p = p0 + 16 * m + (lane & 15);
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = acc[j][m][i] + bv[i];
      if constexpr (EPI == SPS_NN_EPI_PLAIN) {
        const int64_t o = (int64_t)p * K + ch;
        if (pre) store4(pre + o, v);
        if (act) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = silu(v[i]);
        }
        store4(y + o, v);
      } else {
        const int n = pn[m], hh = ph[m], ww = pw[m];
#pragma unroll
        for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
          for (int b2 = 0; b2 < 2; ++b2) {
            const int64_t o =
                ((int64_t)(n * 2 * H + 2 * hh + a2) * (2 * W) + 2 * ww + b2) * K +
                ch;
            float u[4];
            load4(skip + o, u);
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] += v[i];
            if (pre) store4(pre + o, u);
            if (act) {
#pragma unroll
              for (int i = 0; i < 4; ++i) u[i] = silu(u[i]);
            }
            store4(y + o, u);
          }
      }
    }
  }
}

// Forward on spatial tiles staged in LDS.  A workgroup owns TH = NW*WN rows
// x 16 columns of one image and KB = 16*MW*WM output channels; the 4 waves
// split that WM x WN ways, each wave holding MW x NW accumulator tiles
// (16 channels x 16 pixels each, one N tile = 16 columns of one row).  Per
// 32-channel chunk of the input the tile plus its 1-pixel periodic halo,
// (TH+2) x 18 pixels, is copied to LDS once (double-buffered across chunks)
// and the 9 taps read their shifted B fragments from there: each activation
// value leaves HBM/L2 once per chunk instead of once per tap.  A fragments
// (weights, [tap][out][in]) are 16-byte global loads that every workgroup
// shares through L2.  A pixel's 32 channels are padded to 40 in LDS so the
// 16 pixels of one fragment start 20 banks apart.
// NCH > 0 (C = 32 * NCH input channels) stages every chunk at once, one LDS
// buffer per chunk, before the taps: the staging registers are free by then,
// which lets a CU hold more workgroups.  NCH = 0 loops over C / 32 chunks
// with two buffers, fetching the next chunk during the current one's taps.
constexpr int kTileCols = 16;
constexpr int kHaloCols = kTileCols + 2;
constexpr int kPixStride = 40;  // bf16 per staged pixel (32 channels + pad)

template <int MW, int NW, int WM, int WN, int EPI, int NCH>
__global__ __launch_bounds__(256) void conv_fwd_tile(
    const uint16_t* __restrict__ x, int N, int H, int W, int C,
    const uint16_t* __restrict__ wt, const float* __restrict__ bias, int K,
    int act, const uint16_t* __restrict__ skip, uint16_t* __restrict__ y,
    uint16_t* __restrict__ pre) {
  constexpr int TH = NW * WN;
  constexpr int KB = 16 * MW * WM;
  constexpr int TILE = (TH + 2) * kHaloCols;        // staged pixels
  constexpr int PIECES = TILE * 4;                  // 16-byte pieces per chunk
  constexpr int PER_THREAD = (PIECES + 255) / 256;
  // Epilogue through LDS when the block's FP32 results fit 40 KiB: the
  // workgroup then writes whole runs of pixels x channels per store (the
  // accumulator layout gives each lane 4 channels of one pixel, 8 bytes)
  constexpr int SKB = KB + 4;  // staged pixel stride: float4 writes of 16
                               // pixels start 16 bytes x 9 apart (no conflicts)
  constexpr int OUT_FLOATS = TH * kTileCols * SKB;
  constexpr bool STAGED = OUT_FLOATS * 4 <= 40960;
  constexpr int NBUF = NCH == 0 ? 2 : NCH;
  constexpr int TILE_BYTES = NBUF * TILE * kPixStride * 2;
  constexpr int LDS_BYTES =
      STAGED && OUT_FLOATS * 4 > TILE_BYTES ? OUT_FLOATS * 4 : TILE_BYTES;
  __shared__ __align__(16) unsigned char lds[LDS_BYTES];
  uint16_t(*tile)[TILE * kPixStride] =
      reinterpret_cast<uint16_t(*)[TILE * kPixStride]>(lds);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int tiles_w = W / kTileCols, tiles_h = H / TH;
  // neighbouring tiles, which share halo pixels, on one XCD
  int t = xcd_remap(blockIdx.x, gridDim.x);
  const int tw = t % tiles_w;
  t /= tiles_w;
  const int th = t % tiles_h;
  const int n = t / tiles_h;
  const int h0 = th * TH, w0 = tw * kTileCols;
  const int k0 = blockIdx.y * KB + 16 * MW * wm;
  const int cq = (lane >> 4) * 8;

  // global source offsets of this thread's staging pieces (channel 0)
  int64_t src[PER_THREAD];
  int dst[PER_THREAD];
#pragma unroll
  for (int i = 0; i < PER_THREAD; ++i) {
    const int e = threadIdx.x + 256 * i;
    const int pix = e >> 2, q = e & 3;
    const int tr = pix / kHaloCols, tc = pix - tr * kHaloCols;
    const int row = wrapi(h0 + tr - 1, H), col = wrapi(w0 + tc - 1, W);
    src[i] = e < PIECES ? ((int64_t)(n * H + row) * W + col) * C + 8 * q : -1;
    dst[i] = pix * kPixStride + 8 * q;
  }
  constexpr int NST = NCH > 1 ? NCH : 1;  // staging register sets
  u32x4 stage[NST][PER_THREAD];
  auto fetch = [&](int c0, int k) {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i)
      if (src[i] >= 0)
        stage[k][i] = *reinterpret_cast<const u32x4*>(x + src[i] + c0);
  };
  auto put = [&](int buf, int k) {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i)
      if (src[i] >= 0)
        *reinterpret_cast<u32x4*>(&tile[buf][dst[i]]) = stage[k][i];
  };

  f32x4v acc[MW][NW];
#pragma unroll
  for (int m = 0; m < MW; ++m)
#pragma unroll
    for (int j = 0; j < NW; ++j) acc[m][j] = f32x4v{0.f, 0.f, 0.f, 0.f};

  const int nchunks = NCH ? NCH : C / 32;
  // NCH > 0: every chunk's loads in flight before the first LDS store
#pragma unroll
  for (int c = 0; c < NST; ++c) fetch(32 * c, c);
  // With one chunk and 32 channels per wave the weights of all nine taps fit
  // the registers (72) at three waves per SIMD: one latency instead of nine
  // (32->32 at 256^2, batch 64: 190 -> 167 us).
  constexpr bool ALLW = NCH == 1 && MW == 2;
  bf16x8 aw[ALLW ? 9 : 1][MW];
  if constexpr (ALLW) {
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
      for (int m = 0; m < MW; ++m)
        aw[tap][m] = load_frag(wt + ((int64_t)tap * K + k0 + 16 * m + (lane & 15)) * C + cq);
  }
#pragma unroll
  for (int c = 0; c < NST; ++c) put(c, c);
  for (int ch = 0; ch < nchunks; ++ch) {
    const int buf = NCH ? ch : ch & 1;
    const int c0 = 32 * ch;
    // otherwise weight fragments are loaded one tap ahead of their MFMAs
    // (loading all nine taps' at once costs the waves a SIMD can hold)
    bf16x8 apre[2][MW];
    auto load_a = [&](int tap, bf16x8 (&dst)[MW]) {
#pragma unroll
      for (int m = 0; m < MW; ++m)
        dst[m] = load_frag(wt + ((int64_t)tap * K + k0 + 16 * m + (lane & 15)) * C +
                           c0 + cq);
    };
    if constexpr (!ALLW) load_a(0, apre[0]);
    // NCH = 0: tile[buf] written and tile[buf ^ 1] free; NCH > 0: every
    // chunk's tile written
    if (NCH == 0 || ch == 0) __syncthreads();
    if (NCH == 0 && ch + 1 < nchunks) fetch(32 * (ch + 1), 0);
    const uint16_t* tb = tile[buf];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      const int dr = tap / 3, ds = tap % 3;  // halo-shifted offsets 0..2
      bf16x8 b[NW];
      if constexpr (!ALLW)
        if (tap + 1 < 9) load_a(tap + 1, apre[(tap + 1) & 1]);
      const bf16x8 (&a)[MW] = ALLW ? aw[ALLW ? tap : 0] : apre[tap & 1];
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        const int tr = wn * NW + j + dr;
        const int tc = (lane & 15) + ds;
        b[j] = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u32x4*>(
                        tb + (tr * kHaloCols + tc) * kPixStride + cq));
      }
#pragma unroll
      for (int m = 0; m < MW; ++m)
#pragma unroll
        for (int j = 0; j < NW; ++j)
          acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[j],
                                                              acc[m][j], 0, 0, 0);
    }
    if (NCH == 0 && ch + 1 < nchunks) put(buf ^ 1, 0);
  }

  if constexpr (STAGED) {
    // stage[pixel][channel] in FP32, pixel = row * 16 + column of the tile
    float* stage = reinterpret_cast<float*>(lds);
    const int kb0 = blockIdx.y * KB;
    __syncthreads();  // every wave is done with the input tile
#pragma unroll
    for (int m = 0; m < MW; ++m) {
      const int cl = 16 * MW * wm + 16 * m + 4 * (lane >> 4);
      float bv[4] = {0.f, 0.f, 0.f, 0.f};
      if (bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bv[i] = bias[kb0 + cl + i];
      }
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        const int px = (wn * NW + j) * kTileCols + (lane & 15);
        *reinterpret_cast<f32x4v*>(&stage[px * SKB + cl]) =
            f32x4v{acc[m][j][0] + bv[0], acc[m][j][1] + bv[1], acc[m][j][2] + bv[2],
                   acc[m][j][3] + bv[3]};
      }
    }
    __syncthreads();
    constexpr int G = KB / 8;  // 8-channel groups per pixel
    if constexpr (EPI == SPS_NN_EPI_PLAIN) {
      for (int e = threadIdx.x; e < TH * kTileCols * G; e += 256) {
        const int px = e / G, g = e - px * G;
        const int hh = h0 + px / kTileCols, ww = w0 + px % kTileCols;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = stage[px * SKB + 8 * g + i];
        const int64_t o = ((int64_t)(n * H + hh) * W + ww) * K + kb0 + 8 * g;
        if (pre) store8(pre + o, v);
        if (act) {
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = silu(v[i]);
        }
        store8(y + o, v);
      }
    } else {
      // output (2*TH) x 32 pixels, each from tile pixel (r/2, c/2); the
      // skip pieces of U iterations are loaded before any is used, so their
      // memory latencies overlap instead of adding up
      constexpr int ITERS = 4 * TH * kTileCols * G / 256;
      static_assert(4 * TH * kTileCols * G % 256 == 0, "whole iterations");
      constexpr int U = ITERS % 4 == 0 ? 4 : 1;
      for (int it = 0; it < ITERS; it += U) {
        int64_t o[U];
        int sp[U];
        float u[U][8];
#pragma unroll
        for (int q = 0; q < U; ++q) {
          const int e = threadIdx.x + 256 * (it + q);
          const int opx = e / G, g = e - opx * G;
          const int orow = opx / (2 * kTileCols), ocol = opx % (2 * kTileCols);
          sp[q] = ((orow >> 1) * kTileCols + (ocol >> 1)) * SKB + 8 * g;
          o[q] = ((int64_t)(n * 2 * H + 2 * h0 + orow) * (2 * W) + 2 * w0 + ocol) * K +
                 kb0 + 8 * g;
          load8(skip + o[q], u[q]);
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
#pragma unroll
          for (int i = 0; i < 8; ++i) u[q][i] += stage[sp[q] + i];
          if (pre) store8(pre + o[q], u[q]);
          if (act) {
#pragma unroll
            for (int i = 0; i < 8; ++i) u[q][i] = silu(u[q][i]);
          }
          store8(y + o[q], u[q]);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < MW; ++m) {
    const int chn = k0 + 16 * m + 4 * (lane >> 4);  // 4 consecutive channels
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
      for (int i = 0; i < 4; ++i) bv[i] = bias[chn + i];
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const int hh = h0 + wn * NW + j, ww = w0 + (lane & 15);
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = acc[m][j][i] + bv[i];
      if constexpr (EPI == SPS_NN_EPI_PLAIN) {
        const int64_t o = ((int64_t)(n * H + hh) * W + ww) * K + chn;
        if (pre) store4(pre + o, v);
        if (act) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = silu(v[i]);
        }
        store4(y + o, v);
      } else {
#pragma unroll
        for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
          for (int b2 = 0; b2 < 2; ++b2) {
            const int64_t o =
                ((int64_t)(n * 2 * H + 2 * hh + a2) * (2 * W) + 2 * ww + b2) * K +
                chn;
            float u[4];
            load4(skip + o, u);
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] += v[i];
            if (pre) store4(pre + o, u);
            if (act) {
#pragma unroll
              for (int i = 0; i < 4; ++i) u[i] = silu(u[i]);
            }
            store4(y + o, u);
          }
      }
    }
  }
}

// The plain epilogue of a workgroup: bias and activation on the accumulators,
// rounded to BF16, then through LDS (pixel stride KB + 8) so that stores are
// runs of pixels x channels in 16-byte pieces.  acc[m][j] holds channels
// cl + 16*m .. + 3 of pixel px + 16*j of the tile (16 columns per row).  pre,
// when asked for, goes the same way first.  (With the FP32 sums staged and
// activated after the read, twice the LDS bytes, 64->64 took 133 us, not 125.)
template <int KB, int NPX, int NT, int MW, int NW>
__device__ __forceinline__ void store_plain(
    f32x4v (&acc)[MW][NW], uint16_t* stage, int px, int cl,
    const float* __restrict__ bias, int act, uint16_t* __restrict__ y,
    uint16_t* __restrict__ pre, int64_t base, int W, int K) {
  constexpr int S = KB + 8, G = KB / 8;
  if (bias) {
#pragma unroll
    for (int m = 0; m < MW; ++m) {
      f32x4v b;
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = bias[cl + 16 * m + i];
#pragma unroll
      for (int j = 0; j < NW; ++j) acc[m][j] += b;
    }
  }
  auto pass = [&](uint16_t* out, bool silu_it) {
    __syncthreads();  // the workgroup is done with what the LDS held
#pragma unroll
    for (int m = 0; m < MW; ++m)
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = silu_it ? silu(acc[m][j][i]) : acc[m][j][i];
        store4(&stage[(px + 16 * j) * S + cl + 16 * m], v);
      }
    __syncthreads();
#pragma unroll
    for (int e0 = 0; e0 < NPX * G; e0 += NT) {
      const int e = e0 + threadIdx.x;
      if (NPX * G % NT != 0 && e >= NPX * G) break;
      const int q = e / G, g = e - q * G;
      *reinterpret_cast<u32x4*>(out + base + ((int64_t)(q / kTileCols) * W + q % kTileCols) * K +
                                8 * g) =
          *reinterpret_cast<const u32x4*>(&stage[q * S + 8 * g]);
    }
  };
  if (pre) pass(pre, false);
  pass(y, act != 0);
}

// Forward on large tiles, 8 waves: TH = 4*WN rows x 16 columns by KB = 64*WM
// output channels, each wave 64 channels x 64 pixels.  conv_fwd_tile's waves
// wait 83% of their time on weights: every wave reads its own fragments from
// L2 (1.2 GB per call of 256->256 at 32^2, batch 64, for 1.2 MB of weights),
// and the products keep the matrix cores busy 20% of the time.  Here a
// workgroup stages the weights of three taps of a 32-channel chunk in LDS, in
// fragment order, double-buffered like the input tile, with the next group's
// loads in flight during this group's 48 products per wave, so a weight is
// read once per 256 or 512 pixels.  Products and sums are those of
// conv_fwd_tile in the same order.  Bound by LDS reads and barriers now: 40% of
// the matrix cores' rate at 256 channels.  Measured (us, batch 64, before ->
// now): 64->64 at 128^2 187 -> 125; 128->128 at 64^2 153 -> 96; 256->256 at
// 32^2 144 -> 80 (960 TFLOP/s); upsample-add 256->128 149 -> 57, 128->64 181 ->
// 89.
template <int WM, int WN, int EPI>
__global__ __launch_bounds__(512) void conv_fwd_wide(
    const uint16_t* __restrict__ x, int H, int W, int C,
    const uint16_t* __restrict__ wt, const float* __restrict__ bias, int K,
    int act, const uint16_t* __restrict__ skip, uint16_t* __restrict__ y,
    uint16_t* __restrict__ pre) {
  static_assert(WM * WN == 8, "8 waves");
  constexpr int NT = 512, MW = 4, NW = 4;
  constexpr int TH = NW * WN, KB = 16 * MW * WM;
  constexpr int TILE = (TH + 2) * kHaloCols;
  constexpr int TP = TILE * 4, NTP = (TP + NT - 1) / NT;    // tile pieces
  constexpr int WPC = 3 * KB * 4, NWP = (WPC + NT - 1) / NT;  // weight pieces
  constexpr int kTile = TILE * kPixStride, kW = 3 * KB * 32;
  constexpr int SKB = KB + 4;                 // staged pixel stride (FP32)
  constexpr int PXH = TH * kTileCols / 2;     // pixels of an epilogue pass
  constexpr int kMain = 2 * (kTile + kW) * 2;
  constexpr int kEpi = EPI == SPS_NN_EPI_PLAIN ? TH * kTileCols * (KB + 8) * 2 : PXH * SKB * 4;
  __shared__ __align__(16) unsigned char lds[kMain > kEpi ? kMain : kEpi];
  uint16_t* const tiles = reinterpret_cast<uint16_t*>(lds);
  uint16_t* const weights = tiles + 2 * kTile;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int cq = (lane >> 4) * 8;
  // output-channel blocks of one tile are neighbours, on one XCD
  const int nkb = K / KB;
  int t = xcd_remap(blockIdx.x, gridDim.x);
  const int kb0 = t % nkb * KB;
  t /= nkb;
  const int tiles_w = W / kTileCols, tiles_h = H / TH;
  const int w0 = t % tiles_w * kTileCols;
  t /= tiles_w;
  const int h0 = t % tiles_h * TH, n = t / tiles_h;

  int64_t src[NTP];
#pragma unroll
  for (int i = 0; i < NTP; ++i) {
    const int e = threadIdx.x + NT * i, pix = e >> 2, q = e & 3;
    const int tr = pix / kHaloCols, tc = pix - tr * kHaloCols;
    const int row = wrapi(h0 + tr - 1, H), col = wrapi(w0 + tc - 1, W);
    src[i] = e < TP ? ((int64_t)(n * H + row) * W + col) * C + 8 * q : -1;
  }
  u32x4 rt[NTP], rw[NWP];
  auto fetch_tile = [&](int c0) {
#pragma unroll
    for (int i = 0; i < NTP; ++i)
      if (src[i] >= 0) rt[i] = *reinterpret_cast<const u32x4*>(x + src[i] + c0);
  };
  auto put_tile = [&](int b) {
#pragma unroll
    for (int i = 0; i < NTP; ++i) {
      const int e = threadIdx.x + NT * i;
      if (src[i] >= 0)
        *reinterpret_cast<u32x4*>(tiles + b * kTile + (e >> 2) * kPixStride + 8 * (e & 3)) = rt[i];
    }
  };
  // group g: taps 3*(g % 3) .. + 2 of chunk g / 3; piece e is lane e % 64's
  // fragment of channel tile e / 64
  auto fetch_w = [&](int g) {
    const int tap0 = 3 * (g % 3), c0 = 32 * (g / 3);
#pragma unroll
    for (int i = 0; i < NWP; ++i) {
      const int e = threadIdx.x + NT * i;
      const int tap = e / (KB * 4), r = e % (KB * 4), l = r & 63;
      if (WPC % NT == 0 || e < WPC)
        rw[i] = *reinterpret_cast<const u32x4*>(
            wt + ((int64_t)(tap0 + tap) * K + kb0 + (r >> 6) * 16 + (l & 15)) * C + c0 +
            8 * (l >> 4));
    }
  };
  auto put_w = [&](int b) {
#pragma unroll
    for (int i = 0; i < NWP; ++i) {
      const int e = threadIdx.x + NT * i;
      if (WPC % NT == 0 || e < WPC)
        *reinterpret_cast<u32x4*>(weights + b * kW + 8 * e) = rw[i];
    }
  };

  f32x4v acc[MW][NW];
#pragma unroll
  for (int m = 0; m < MW; ++m)
#pragma unroll
    for (int j = 0; j < NW; ++j) acc[m][j] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const int nchunks = C / 32;
  fetch_tile(0);
  fetch_w(0);
  put_tile(0);
  put_w(0);
  __syncthreads();
  for (int ch = 0; ch < nchunks; ++ch) {
    const uint16_t* tb = tiles + (ch & 1) * kTile;
    const bool more = ch + 1 < nchunks;
#pragma unroll
    for (int dr = 0; dr < 3; ++dr) {
      const int g = 3 * ch + dr;
      if (dr < 2 || more) fetch_w(g + 1);
      if (dr == 0 && more) fetch_tile(32 * (ch + 1));
      const uint16_t* wb = weights + (g & 1) * kW + 8 * lane;
#pragma unroll
      for (int ds = 0; ds < 3; ++ds) {
        bf16x8 a[MW], b[NW];
#pragma unroll
        for (int m = 0; m < MW; ++m)
          a[m] = __builtin_bit_cast(
              bf16x8, *reinterpret_cast<const u32x4*>(
                          wb + ((ds * (KB / 16)) + wm * MW + m) * 512));
#pragma unroll
        for (int j = 0; j < NW; ++j)
          b[j] = __builtin_bit_cast(
              bf16x8, *reinterpret_cast<const u32x4*>(
                          tb + ((wn * NW + j + dr) * kHaloCols + (lane & 15) + ds) * kPixStride +
                          cq));
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
          for (int j = 0; j < NW; ++j)
            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[j], acc[m][j], 0, 0, 0);
      }
      if (dr < 2 || more) put_w((g + 1) & 1);
      if (dr == 2 && more) put_tile((ch + 1) & 1);
      __syncthreads();
    }
  }

  if constexpr (EPI == SPS_NN_EPI_PLAIN) {
    store_plain<KB, TH * kTileCols, NT>(
        acc, reinterpret_cast<uint16_t*>(lds), wn * NW * kTileCols + (lane & 15),
        16 * MW * wm + 4 * (lane >> 4), bias ? bias + kb0 : nullptr, act, y, pre,
        ((int64_t)(n * H + h0) * W + w0) * K + kb0, W, K);
    return;
  }
  // upsample-add epilogue through LDS, half of the rows at a time: FP32 sums
  // with the bias, then runs of pixels x channels in 16-byte pieces
  float* stage = reinterpret_cast<float*>(lds);
  constexpr int G = KB / 8;
  for (int half = 0; half < 2; ++half) {
    if (wn / (WN / 2) == half) {
#pragma unroll
      for (int m = 0; m < MW; ++m) {
        const int cl = 16 * (MW * wm + m) + 4 * (lane >> 4);
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias) {
#pragma unroll
          for (int i = 0; i < 4; ++i) bv[i] = bias[kb0 + cl + i];
        }
#pragma unroll
        for (int j = 0; j < NW; ++j) {
          const int px = (wn % (WN / 2) * NW + j) * kTileCols + (lane & 15);
          *reinterpret_cast<f32x4v*>(&stage[px * SKB + cl]) =
              f32x4v{acc[m][j][0] + bv[0], acc[m][j][1] + bv[1], acc[m][j][2] + bv[2],
                     acc[m][j][3] + bv[3]};
        }
      }
    }
    __syncthreads();
    const int hb = h0 + half * (TH / 2);
    {
      constexpr int ITERS = 4 * PXH * G / NT, U = 4;
      static_assert(ITERS % U == 0, "whole iterations");
      for (int it = 0; it < ITERS; it += U) {
        int64_t o[U];
        int sp[U];
        float u[U][8];
#pragma unroll
        for (int q = 0; q < U; ++q) {
          const int e = threadIdx.x + NT * (it + q);
          const int opx = e / G, g = e - opx * G;
          const int orow = opx / (2 * kTileCols), ocol = opx % (2 * kTileCols);
          sp[q] = ((orow >> 1) * kTileCols + (ocol >> 1)) * SKB + 8 * g;
          o[q] = ((int64_t)(n * 2 * H + 2 * hb + orow) * (2 * W) + 2 * w0 + ocol) * K + kb0 +
                 8 * g;
          load8(skip + o[q], u[q]);
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
#pragma unroll
          for (int i = 0; i < 8; ++i) u[q][i] += stage[sp[q] + i];
          if (pre) store8(pre + o[q], u[q]);
          if (act) {
#pragma unroll
            for (int i = 0; i < 8; ++i) u[q][i] = silu(u[q][i]);
          }
          store8(y + o[q], u[q]);
        }
      }
    }
    __syncthreads();
  }
}

// Weight gradient (and bias gradient) on blocks of pixels: a workgroup owns a
// KT x CT tile of [k][c] for all 9 taps and walks chunks of RC rows x WC
// columns.  Per chunk dpre and the input with its 1-pixel periodic halo are
// copied to LDS (two buffers, the next chunk's loads in flight during this
// one's products).  Both operands need consecutive pixels of one channel per
// lane while LDS rows are consecutive channels of one pixel:
// ds_read_b64_tr_b16 transposes 4 pixels x 16 channels per 16 lanes.  The
// three horizontal taps come from one read of 12 pixels, shifted in registers.
// Each of the 8 waves holds a 32 x 32 part of the tile (144 accumulators) and
// the WP waves of a part split the chunk's pixels; their sums are added in
// order at the end.  Rows are padded so that the 4 pixels of a read fall in
// different banks.
// The form that gathered fragments with 2-byte LDS reads and staged 32 pixels
// at a time took (batch 32) 128 us for 32->32 at 256^2 and 94 on average for
// the layers of 64 channels and more; this one 75 and 40 (with the sum over
// workgroups 470 and 600 TFLOP/s), the bias gradient included, which was a
// pass over dpre of its own (37 us on average).
typedef short i16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 read_tr(const uint16_t* p) {
  return __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 (__attribute__((address_space(3))) i16x4*)p));
}

__device__ __forceinline__ bf16x8 bf16_ones() {
  constexpr uint32_t kOnes = 0x3f803f80u;  // two BF16 ones
  return __builtin_bit_cast(bf16x8, u32x4{kOnes, kOnes, kOnes, kOnes});
}

template <int KT, int CT, int WC>
struct WgradTile {
  static constexpr int kThreads = 512;
  static constexpr int WK = KT / 32, WCT = CT / 32;  // parts of the tile
  static constexpr int WP = 8 / (WK * WCT);          // waves of a part
  static constexpr int PX = WP == 8 ? 256 : 128;     // pixels of a chunk
  static constexpr int KS = PX / 32 / WP;            // MFMA steps of a wave
  static constexpr int RC = PX / WC;                 // rows of a chunk
  static constexpr int XC = WC + 4;  // halo, and 2 columns only read past it
  static constexpr int SD = KT + (KT == 64 ? 8 : 16);  // row strides
  static constexpr int SX = CT + (CT == 64 ? 8 : 16);
  static constexpr int kDy = PX * SD, kX = (RC + 2) * XC * SX;
  static constexpr int kBuf = kDy + kX;
};

template <int KT, int CT, int WC>
__global__ __launch_bounds__(512) void conv_wgrad_tile(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy, int H,
    int W, int C, int K, float* __restrict__ part, int64_t slice, int nchunks,
    int per, int with_bias) {
  using G = WgradTile<KT, CT, WC>;
  constexpr int NT = G::kThreads;
  __shared__ __align__(16) uint16_t lds[2 * G::kBuf];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wk = wave % G::WK, wc = wave / G::WK % G::WCT,
            wp = wave / (G::WK * G::WCT);
  const int c0 = blockIdx.x * CT, k0 = blockIdx.y * KT;
  const int cblocks = W / WC, rblocks = H / G::RC;

  constexpr int DP = G::PX * KT / 8, XP = (G::RC + 2) * (WC + 2) * CT / 8;
  constexpr int ND = (DP + NT - 1) / NT, NX = (XP + NT - 1) / NT;
  u32x4 rd[ND], rx[NX];
  auto fetch = [&](int ch) {
    const int cb = ch % cblocks, t = ch / cblocks;
    const int h0 = t % rblocks * G::RC, n = t / rblocks, w0 = cb * WC;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int e = threadIdx.x + NT * i;
      const int px = e / (KT / 8), k = e % (KT / 8) * 8;
      if (DP % NT == 0 || e < DP)
        rd[i] = *reinterpret_cast<const u32x4*>(
            dy + ((int64_t)(n * H + h0 + px / WC) * W + w0 + px % WC) * K + k0 + k);
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = threadIdx.x + NT * i;
      const int px = e / (CT / 8), c = e % (CT / 8) * 8;
      const int r = px / (WC + 2), q = px % (WC + 2);
      if (XP % NT == 0 || e < XP)
        rx[i] = *reinterpret_cast<const u32x4*>(
            x + ((int64_t)(n * H + wrapi(h0 + r - 1, H)) * W + wrapi(w0 + q - 1, W)) * C +
            c0 + c);
    }
  };
  auto put = [&](uint16_t* b) {
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int e = threadIdx.x + NT * i;
      const int px = e / (KT / 8), k = e % (KT / 8) * 8;
      if (DP % NT == 0 || e < DP) *reinterpret_cast<u32x4*>(b + px * G::SD + k) = rd[i];
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = threadIdx.x + NT * i;
      const int px = e / (CT / 8), c = e % (CT / 8) * 8;
      const int r = px / (WC + 2), q = px % (WC + 2);
      if (XP % NT == 0 || e < XP)
        *reinterpret_cast<u32x4*>(b + G::kDy + (r * G::XC + q) * G::SX + c) = rx[i];
    }
  };

  f32x4v acc[9][2][2], accb[2];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[t][a][b] = f32x4v{0.f, 0.f, 0.f, 0.f};
  accb[0] = accb[1] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const bool bias_wave = with_bias && blockIdx.x == 0 && wc == 0;

  const int first = blockIdx.z * per, last = min(nchunks, first + per);
  if (first < last) {
    fetch(first);
    put(lds);
  }
  __syncthreads();
  for (int ch = first; ch < last; ++ch) {
    if (ch + 1 < last) fetch(ch + 1);
    const uint16_t* b = lds + ((ch - first) & 1) * G::kBuf;
#pragma unroll
    for (int ks = 0; ks < G::KS; ++ks) {
      // this lane group's 8 pixels, one row's
      const int px = 32 * (wp * G::KS + ks) + 8 * (lane >> 4);
      const int row = px / WC, col = px % WC;
      const int tp = (lane & 15) >> 2, tc4 = 4 * (lane & 3);
      bf16x8 a[2];
#pragma unroll
      for (int tk = 0; tk < 2; ++tk) {
        const uint16_t* q = b + (px + tp) * G::SD + 32 * wk + 16 * tk + tc4;
        const uint2 u = read_tr(q), v = read_tr(q + 4 * G::SD);
        a[tk] = __builtin_bit_cast(bf16x8, u32x4{u.x, u.y, v.x, v.y});
      }
      if (bias_wave) {
#pragma unroll
        for (int tk = 0; tk < 2; ++tk)
          accb[tk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tk], bf16_ones(), accb[tk], 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int tc = 0; tc < 2; ++tc) {
          const uint16_t* q = b + G::kDy + ((row + r) * G::XC + col + tp) * G::SX +
                              32 * wc + 16 * tc + tc4;
          const uint2 u = read_tr(q), v = read_tr(q + 4 * G::SX), w = read_tr(q + 8 * G::SX);
          const uint32_t d[5] = {u.x, u.y, v.x, v.y, w.x};  // pixels 0 .. 9
          u32x4 f[3];
          f[0] = u32x4{d[0], d[1], d[2], d[3]};
          f[2] = u32x4{d[1], d[2], d[3], d[4]};
#pragma unroll
          for (int i = 0; i < 4; ++i) f[1][i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], 16);
#pragma unroll
          for (int s3 = 0; s3 < 3; ++s3)
#pragma unroll
            for (int tk = 0; tk < 2; ++tk)
              acc[3 * r + s3][tk][tc] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  a[tk], __builtin_bit_cast(bf16x8, f[s3]), acc[3 * r + s3][tk][tc], 0, 0, 0);
        }
    }
    if (ch + 1 < last) put(lds + ((ch + 1 - first) & 1) * G::kBuf);
    __syncthreads();
  }

  // add the WP waves of each part in order through LDS, a tap row at a time,
  // then the bias sums
  if constexpr (G::WP > 1) {
    constexpr int PARTS = G::WK * G::WCT;
    static_assert((G::WP - 1) * PARTS * 64 * 12 * 16 <= 2 * G::kBuf * 2, "fits");
    f32x4v* red = reinterpret_cast<f32x4v*>(lds);
    auto slot = [&](int p) { return red + ((p - 1) * PARTS + wk + G::WK * wc) * 12 * 64 + lane; };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (wp > 0) {
        f32x4v* o = slot(wp);
#pragma unroll
        for (int i = 0; i < (r < 3 ? 12 : 2); ++i)
          o[64 * i] = r < 3 ? acc[3 * (r % 3) + i / 4][i / 2 % 2][i % 2] : accb[i % 2];
      }
      __syncthreads();
      if (wp == 0) {
        for (int p = 1; p < G::WP; ++p) {
          const f32x4v* o = slot(p);
#pragma unroll
          for (int i = 0; i < (r < 3 ? 12 : 2); ++i) {
            if (r < 3) acc[3 * (r % 3) + i / 4][i / 2 % 2][i % 2] += o[64 * i];
            else accb[i % 2] += o[64 * i];
          }
        }
      }
      __syncthreads();
    }
  }
  if (wp > 0) return;
  // this workgroup's partial sums (zeros if it had no chunk)
  float* dw = part + (int64_t)blockIdx.z * slice;
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int tk = 0; tk < 2; ++tk)
#pragma unroll
      for (int tc = 0; tc < 2; ++tc)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = k0 + 32 * wk + 16 * tk + 4 * (lane >> 4) + i;
          const int c = c0 + 32 * wc + 16 * tc + (lane & 15);
          dw[((int64_t)tap * K + k) * C + c] = acc[tap][tk][tc][i];
        }
  if (bias_wave && (lane & 15) == 0) {
#pragma unroll
    for (int tk = 0; tk < 2; ++tk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dw[(int64_t)9 * K * C + k0 + 32 * wk + 16 * tk + 4 * (lane >> 4) + i] = accb[tk][i];
  }
}

// The general weight gradient, for images that do not split into whole chunks
// of the tiled one: tile KT x CT of [k][c] for all 9 taps, reduction over
// 32-pixel row chunks staged in LDS.  Wave w owns k rows [w%2 * KT/2, +KT/2)
// and c columns [w/2 * CT/2, +CT/2).
// ROWS: chunks are 32-pixel pieces of one row (w % 32 == 0) and the three
// input rows with a 1-column halo are staged once; otherwise chunks are any
// 32 consecutive pixels and the nine shifted pixels are staged per tap.
// The bias gradient is a product of the staged dpre with ones, in two waves of
// the first column of workgroups.  Layers of 256 channels, 56 images of 24^2
// and 20 of 40^2, both gradients: 195 and 184 us; with a library sum of dpre
// 227 and 216, with a kernel of one thread per channel 473 and 461.
template <int KT, int CT, bool ROWS>
__global__ __launch_bounds__(256) void conv_wgrad(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy, int N,
    int H, int W, int C, int K, float* __restrict__ part, int64_t slice,
    int nchunks, int chunks_per_block, int with_bias) {
  constexpr int TK = KT / 32, TC = CT / 32;  // MFMA tiles per wave
  __shared__ __align__(16) uint16_t sdy[32][KT + 2];
  __shared__ __align__(16) uint16_t sx[ROWS ? 3 : 9][ROWS ? 34 : 32][CT + 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = blockIdx.x * CT, k0 = blockIdx.y * KT;
  const int kw = (wave & 1) * (KT / 2), cw = (wave >> 1) * (CT / 2);
  const int rowchunks = W / 32;
  f32x4v acc[9][TK][TC];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int a = 0; a < TK; ++a)
#pragma unroll
      for (int b = 0; b < TC; ++b) acc[t][a][b] = f32x4v{0.f, 0.f, 0.f, 0.f};
  f32x4v accb[TK];
#pragma unroll
  for (int a = 0; a < TK; ++a) accb[a] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const bool bias_wave = with_bias && blockIdx.x == 0 && wave < 2;

  const int first = blockIdx.z * chunks_per_block;
  const int last = min(nchunks, first + chunks_per_block);
  for (int ch = first; ch < last; ++ch) {
    __syncthreads();
    // staging in pieces of 8 channels: one 16-byte global load, written to
    // the padded LDS row as four 32-bit stores (rows are 4-byte aligned)
    auto put8 = [](uint16_t* dst, const uint16_t* src) {
      const u32x4 q = *reinterpret_cast<const u32x4*>(src);
      uint32_t* d = reinterpret_cast<uint32_t*>(dst);
      d[0] = q.x;
      d[1] = q.y;
      d[2] = q.z;
      d[3] = q.w;
    };
    if constexpr (ROWS) {
      const int n = ch / (H * rowchunks);
      const int rem = ch - n * H * rowchunks;
      const int h = rem / rowchunks;
      const int w0 = (rem - h * rowchunks) * 32;
      // stage dy: 32 pixels x KT channels
      for (int e = threadIdx.x; e < 32 * (KT / 8); e += 256) {
        const int px = e / (KT / 8), k = (e - px * (KT / 8)) * 8;
        put8(&sdy[px][k], dy + ((int64_t)(n * H + h) * W + w0 + px) * K + k0 + k);
      }
      // stage x: rows h-1..h+1, columns w0-1..w0+32, CT channels
      for (int e = threadIdx.x; e < 3 * 34 * (CT / 8); e += 256) {
        const int r = e / (34 * (CT / 8));
        const int e2 = e - r * 34 * (CT / 8);
        const int col = e2 / (CT / 8), c = (e2 - col * (CT / 8)) * 8;
        const int hh = wrapi(h + r - 1, H), ww = wrapi(w0 + col - 1, W);
        put8(&sx[r][col][c], x + ((int64_t)(n * H + hh) * W + ww) * C + c0 + c);
      }
    } else {
      const int64_t pbase = (int64_t)ch * 32;
      for (int e = threadIdx.x; e < 32 * (KT / 8); e += 256) {
        const int px = e / (KT / 8), k = (e - px * (KT / 8)) * 8;
        put8(&sdy[px][k], dy + (pbase + px) * K + k0 + k);
      }
      const int HW = H * W;
      for (int e = threadIdx.x; e < 9 * 32 * (CT / 8); e += 256) {
        const int t = e / (32 * (CT / 8));
        const int e2 = e - t * 32 * (CT / 8);
        const int px = e2 / (CT / 8), c = (e2 - px * (CT / 8)) * 8;
        const int64_t p = pbase + px;
        const int n = (int)(p / HW);
        const int r = (int)(p - (int64_t)n * HW);
        const int h = r / W, w = r - h * W;
        const int hh = wrapi(h + t / 3 - 1, H), ww = wrapi(w + t % 3 - 1, W);
        put8(&sx[t][px][c], x + ((int64_t)(n * H + hh) * W + ww) * C + c0 + c);
      }
    }
    __syncthreads();
    const int pq = (lane >> 4) * 8;
    bf16x8 a[TK];
#pragma unroll
    for (int tk = 0; tk < TK; ++tk) {
      uint16_t v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = sdy[pq + i][kw + 16 * tk + (lane & 15)];
      a[tk] = __builtin_bit_cast(bf16x8, v);
    }
    if (bias_wave) {
#pragma unroll
      for (int tk = 0; tk < TK; ++tk)
        accb[tk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tk], bf16_ones(), accb[tk], 0, 0, 0);
    }
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      const int r = tap / 3, s = tap % 3;
#pragma unroll
      for (int tc = 0; tc < TC; ++tc) {
        uint16_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if constexpr (ROWS)
            v[i] = sx[r][pq + i + s][cw + 16 * tc + (lane & 15)];
          else
            v[i] = sx[tap][pq + i][cw + 16 * tc + (lane & 15)];
        }
        const bf16x8 b = __builtin_bit_cast(bf16x8, v);
#pragma unroll
        for (int tk = 0; tk < TK; ++tk)
          acc[tap][tk][tc] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[tk], b, acc[tap][tk][tc], 0, 0, 0);
      }
    }
  }
  // this block's partial sums (zeros if it had no chunk): slice blockIdx.z
  float* dw = part + (int64_t)blockIdx.z * slice;
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int tk = 0; tk < TK; ++tk)
#pragma unroll
      for (int tc = 0; tc < TC; ++tc)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = k0 + kw + 16 * tk + 4 * (lane >> 4) + i;
          const int c = c0 + cw + 16 * tc + (lane & 15);
          dw[((int64_t)tap * K + k) * C + c] = acc[tap][tk][tc][i];
        }
  if (bias_wave && (lane & 15) == 0) {
#pragma unroll
    for (int tk = 0; tk < TK; ++tk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dw[(int64_t)9 * K * C + k0 + kw + 16 * tk + 4 * (lane >> 4) + i] = accb[tk][i];
  }
}

// ------------------------------------------------------------ thin layers
// The first (1 -> K) and last (K -> 1) convolutions have no GEMM shape; they
// run on the vector units with 16-byte accesses of 8 channels.  K % 8 == 0.

__global__ __launch_bounds__(256) void in1_fwd(const float* __restrict__ x,
                                               int N, int H, int W,
                                               const float* __restrict__ wt,
                                               const float* __restrict__ bias,
                                               int K, int act,
                                               uint16_t* __restrict__ y,
                                               uint16_t* __restrict__ pre) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= (int64_t)N * H * W) return;
  const int HW = H * W;
  const int n = p / HW, r = p - (int64_t)n * HW, h = r / W, w = r - h * W;
  float xv[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
    xv[t] = x[(int64_t)(n * H + wrapi(h + t / 3 - 1, H)) * W +
              wrapi(w + t % 3 - 1, W)];
  for (int k0 = 0; k0 < K; k0 += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float a = bias ? bias[k0 + i] : 0.f;
#pragma unroll
      for (int t = 0; t < 9; ++t) a = fmaf(xv[t], wt[t * K + k0 + i], a);
      v[i] = a;
    }
    if (pre) store8(pre + p * K + k0, v);
    if (act) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = silu(v[i]);
    }
    store8(y + p * K + k0, v);
  }
}

// The same first layer with its stores staged through LDS: each thread
// computes all K channels of one pixel exactly as in1_fwd does (bias, then
// the 9 taps in order, FMA; the weights are uniform across the wave), then
// the workgroup writes its 256 consecutive pixels x K channels, one
// contiguous run, in 16-byte pieces.
template <int K>
__global__ __launch_bounds__(256) void in1_fwd_staged(
    const float* __restrict__ x, int N, int H, int W,
    const float* __restrict__ wt, const float* __restrict__ bias, int act,
    uint16_t* __restrict__ y, uint16_t* __restrict__ pre) {
  __shared__ __align__(16) uint16_t sy[256 * K];
  __shared__ __align__(16) uint16_t sp[256 * K];
  const int64_t np = (int64_t)N * H * W;
  const int64_t p0 = (int64_t)blockIdx.x * 256;
  const int64_t p = p0 + threadIdx.x;
  if (p < np) {
    const int HW = H * W;
    const int n = p / HW, r = p - (int64_t)n * HW, h = r / W, w = r - h * W;
    float xv[9];
#pragma unroll
    for (int t = 0; t < 9; ++t)
      xv[t] = x[(int64_t)(n * H + wrapi(h + t / 3 - 1, H)) * W +
                wrapi(w + t % 3 - 1, W)];
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 8) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float a = bias ? bias[k0 + i] : 0.f;
#pragma unroll
        for (int t = 0; t < 9; ++t) a = fmaf(xv[t], wt[t * K + k0 + i], a);
        v[i] = a;
      }
      if (pre) store8(&sp[threadIdx.x * K + k0], v);
      if (act) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = silu(v[i]);
      }
      store8(&sy[threadIdx.x * K + k0], v);
    }
  }
  __syncthreads();
  const int64_t valid = np - p0 < 256 ? np - p0 : 256;
  const int pieces = (int)valid * K / 8;
  for (int e = threadIdx.x; e < pieces; e += 256) {
    *reinterpret_cast<u32x4*>(y + p0 * K + 8 * e) =
        *reinterpret_cast<const u32x4*>(&sy[8 * e]);
    if (pre)
      *reinterpret_cast<u32x4*>(pre + p0 * K + 8 * e) =
          *reinterpret_cast<const u32x4*>(&sp[8 * e]);
  }
}

// The last layer on 16 x 16 pixel tiles: the tile and its periodic halo
// (18 x 18 pixels x C channels) are staged in LDS once, so each activation
// is read from HBM once instead of once per tap; the weights are uniform
// across the wave.  Same arithmetic order as out1_fwd (bias, then taps, then
// channels in order).
template <int C>
__global__ __launch_bounds__(256) void out1_fwd_tile(
    const uint16_t* __restrict__ x, int N, int H, int W,
    const float* __restrict__ wt, const float* __restrict__ bias,
    float* __restrict__ y) {
  constexpr int T = 16, HT = T + 2;
  constexpr int PS = C + 8;  // padded pixel stride
  __shared__ __align__(16) uint16_t tile[HT * HT * PS];
  const int tiles_w = W / T, tiles_h = H / T;
  int b = blockIdx.x;
  const int tw = b % tiles_w;
  b /= tiles_w;
  const int th = b % tiles_h;
  const int n = b / tiles_h;
  const int h0 = th * T, w0 = tw * T;
  constexpr int groups = C / 8;
  for (int e = threadIdx.x; e < HT * HT * groups; e += 256) {
    const int pix = e / groups, q = e - pix * groups;
    const int tr = pix / HT, tc = pix - tr * HT;
    const int row = wrapi(h0 + tr - 1, H), col = wrapi(w0 + tc - 1, W);
    *reinterpret_cast<u32x4*>(&tile[pix * PS + 8 * q]) =
        *reinterpret_cast<const u32x4*>(x + ((int64_t)(n * H + row) * W + col) * C +
                                        8 * q);
  }
  __syncthreads();
  const int ty = threadIdx.x / T, tx = threadIdx.x % T;
  float v = bias ? bias[0] : 0.f;
  for (int t = 0; t < 9; ++t) {
    const uint16_t* xp = &tile[((ty + t / 3) * HT + tx + t % 3) * PS];
#pragma unroll
    for (int c0 = 0; c0 < C; c0 += 8) {
      float xv[8];
      load8(xp + c0, xv);
#pragma unroll
      for (int i = 0; i < 8; ++i) v = fmaf(xv[i], wt[t * C + c0 + i], v);
    }
  }
  y[(int64_t)(n * H + h0 + ty) * W + w0 + tx] = v;
}

// Weight gradients of the thin layers: part[t][c] = sum_q a[q][c] * s[q'], q'
// the pixel one tap away, (h + dr, w + ds) for SIGN = 1 (the first layer: a the
// gradient, s the input) and (h - dr, w - ds) for SIGN = -1 (the last layer: a
// the input, s the gradient); part[9][c] = sum_q a[q][c], the first layer's
// bias gradient.  A lane is a pixel and keeps the 80 sums of 8 channels in
// registers; a workgroup's 4 waves take neighbouring channels of the same
// pixels, whose cache lines they share.  The lanes are added by halving (each
// step a lane gives away half of its sums).  With a thread per (tap, channel)
// and the pixels in LDS, two reads per product, the two layers took 100 and 115
// us at 32 channels, 256^2, batch 32; this way 43 and 45.
template <int SIGN>
__global__ __launch_bounds__(256) void thin_wgrad(
    const uint16_t* __restrict__ a, const float* __restrict__ s, int64_t np,
    int H, int W, int C, float* __restrict__ part, int64_t slice, int64_t per,
    int with_bias) {
  const int lane = threadIdx.x & 63;
  const int c0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 8;
  if (c0 >= C) return;
  const int64_t p0 = blockIdx.x * per, p1 = min(np, p0 + per);
  const int HW = H * W;
  int64_t p = p0 + lane;
  int64_t img = p / HW;
  int h = (int)(p - img * HW) / W, w = (int)(p - img * HW) - h * W;
  float v[80];
#pragma unroll
  for (int i = 0; i < 80; ++i) v[i] = 0.f;
  for (; p < p1; p += 64) {
    float x[8], sv[9];
    load8(a + p * C + c0, x);
    const float* si = s + img * HW;
    const int hr[3] = {h == 0 ? H - 1 : h - 1, h, h + 1 == H ? 0 : h + 1};
    const int wr[3] = {w == 0 ? W - 1 : w - 1, w, w + 1 == W ? 0 : w + 1};
#pragma unroll
    for (int t = 0; t < 9; ++t)
      sv[t] = si[hr[SIGN > 0 ? t / 3 : 2 - t / 3] * W + wr[SIGN > 0 ? t % 3 : 2 - t % 3]];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int i = 0; i < 8; ++i) v[8 * t + i] = fmaf(sv[t], x[i], v[8 * t + i]);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[72 + i] += x[i];
    for (w += 64; w >= W; w -= W)
      if (++h == H) {
        h = 0;
        ++img;
      }
  }
  int first = 0;  // which of the 80 sums v[0] is
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    const int n = 40 >> st, mask = 32 >> st;
    const bool up = lane & mask;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const float give = up ? v[i] : v[n + i], keep = up ? v[n + i] : v[i];
      v[i] = keep + __shfl_xor(give, mask, 64);
    }
    if (up) first += n;
  }
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    v[i] += __shfl_xor(v[i], 2, 64);
    v[i] += __shfl_xor(v[i], 1, 64);
    const int t = (first + i) / 8, c = c0 + (first + i) % 8;
    if ((lane & 3) == 0 && (t < 9 || with_bias))
      part[blockIdx.x * slice + (int64_t)t * C + c] = v[i];
  }
}

__global__ __launch_bounds__(256) void out1_fwd(const uint16_t* __restrict__ x,
                                                int N, int H, int W, int C,
                                                const float* __restrict__ wt,
                                                const float* __restrict__ bias,
                                                float* __restrict__ y) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= (int64_t)N * H * W) return;
  const int HW = H * W;
  const int n = p / HW, r = p - (int64_t)n * HW, h = r / W, w = r - h * W;
  float v = bias ? bias[0] : 0.f;
  for (int t = 0; t < 9; ++t) {
    const uint16_t* xp =
        x + ((int64_t)(n * H + wrapi(h + t / 3 - 1, H)) * W +
             wrapi(w + t % 3 - 1, W)) * C;
    for (int c0 = 0; c0 < C; c0 += 8) {
      float xv[8];
      load8(xp + c0, xv);
#pragma unroll
      for (int i = 0; i < 8; ++i) v = fmaf(xv[i], wt[t * C + c0 + i], v);
    }
  }
  y[p] = v;
}

// dx[p][c] = sum_t dy[p - shift_t] * w[t][c]
__global__ __launch_bounds__(256) void out1_bwd_data(
    const float* __restrict__ dy, int N, int H, int W, int C,
    const float* __restrict__ wt, uint16_t* __restrict__ dx) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= (int64_t)N * H * W) return;
  const int HW = H * W;
  const int n = p / HW, r = p - (int64_t)n * HW, h = r / W, w = r - h * W;
  float d[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
    d[t] = dy[(int64_t)(n * H + wrapi(h - (t / 3 - 1), H)) * W +
              wrapi(w - (t % 3 - 1), W)];
  for (int c0 = 0; c0 < C; c0 += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float a = 0.f;
#pragma unroll
      for (int t = 0; t < 9; ++t) a = fmaf(d[t], wt[t * C + c0 + i], a);
      v[i] = a;
    }
    store8(dx + p * C + c0, v);
  }
}

// The deterministic sum of M partial gradients of `count` floats each: a
// workgroup takes 64 of the floats, its WAVES waves equal ranges of the partials
// in order, and the ranges are added in order.  The first nw sums go to dw, the
// others (a bias gradient) to db.  The sums are FP64, for the loads set the
// time: added in FP32, the partials of 32 images of 256^2 left the bias gradient
// of positive values off by 6.1e-8 (rel L2), a library's pairwise sum by 3.6e-8;
// this way 2.1e-8.  (Two launches, runs
// of 32 in place first, took 11 + 6 us a layer; one 6.)
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void add_partials(
    const float* __restrict__ part, int M, int64_t count, float* __restrict__ dw,
    int64_t nw, float* __restrict__ db) {
  __shared__ double sh[WAVES][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + lane;
  const int m1 = (int)((int64_t)M * (wave + 1) / WAVES);
  double s = 0.0;
  if (i < count) {
    int m = (int)((int64_t)M * wave / WAVES);
    for (; m + 8 <= m1; m += 8) {
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = part[(int64_t)(m + q) * count + i];
#pragma unroll
      for (int q = 0; q < 8; ++q) s += (double)v[q];
    }
    for (; m < m1; ++m) s += (double)part[(int64_t)m * count + i];
  }
  sh[wave][lane] = s;
  __syncthreads();
  if (wave > 0 || i >= count) return;
  for (int q = 1; q < WAVES; ++q) s += sh[q][lane];
  float* out = i < nw ? dw + i : db + (i - nw);
  *out = (float)((double)*out + s);
}

// ------------------------------------------------------------ elementwise

__global__ __launch_bounds__(256) void silu_bwd_k(const uint16_t* __restrict__ dy,
                                                  const uint16_t* __restrict__ pre,
                                                  uint16_t* __restrict__ dx,
                                                  int64_t count) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * 256) {
    const float z = bf2f(pre[i]);
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
    dx[i] = f2bf(bf2f(dy[i]) * s * (1.0f + z * (1.0f - s)));
  }
}

__global__ __launch_bounds__(256) void pool2_k(const uint16_t* __restrict__ x,
                                               int N, int H, int W, int C,
                                               int mode,
                                               uint16_t* __restrict__ y) {
  const int Ho = H / 2, Wo = W / 2;
  const int64_t total = (int64_t)N * Ho * Wo * C;
  const float scale = mode == 0 ? 0.25f : 1.0f;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * 256) {
    const int c = i % C;
    int64_t q = i / C;
    const int wo = q % Wo;
    q /= Wo;
    const int ho = q % Ho;
    const int n = q / Ho;
    const int64_t b = ((int64_t)(n * H + 2 * ho) * W + 2 * wo) * C + c;
    const float s = (bf2f(x[b]) + bf2f(x[b + C])) +
                    (bf2f(x[b + (int64_t)W * C]) + bf2f(x[b + (int64_t)W * C + C]));
    y[i] = f2bf(s * scale);
  }
}

__global__ __launch_bounds__(256) void unpool2_k(const uint16_t* __restrict__ x,
                                                 int N, int H, int W, int C,
                                                 float scale,
                                                 uint16_t* __restrict__ y) {
  const int Ho = 2 * H, Wo = 2 * W;
  const int64_t total = (int64_t)N * Ho * Wo * C;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * 256) {
    const int c = i % C;
    int64_t q = i / C;
    const int wo = q % Wo;
    q /= Wo;
    const int ho = q % Ho;
    const int n = q / Ho;
    y[i] = f2bf(bf2f(x[((int64_t)(n * H + ho / 2) * W + wo / 2) * C + c]) * scale);
  }
}

// The same three passes on 8 consecutive channels per thread: one 16-byte
// access per operand and 32-bit index arithmetic, used when the channel count
// is a multiple of 8, the piece count fits 31 bits and the pointers are
// 16-byte aligned.  Each value goes through the same operations in the same
// order as in the one-value kernels above, so results are identical.
__global__ __launch_bounds__(256) void silu_bwd_v8(const uint16_t* __restrict__ dy,
                                                   const uint16_t* __restrict__ pre,
                                                   uint16_t* __restrict__ dx,
                                                   unsigned pieces) {
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < pieces; i += gridDim.x * 256) {
    float z[8], d[8], v[8];
    load8(pre + 8 * (int64_t)i, z);
    load8(dy + 8 * (int64_t)i, d);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-z[k]));
      v[k] = d[k] * s * (1.0f + z[k] * (1.0f - s));
    }
    store8(dx + 8 * (int64_t)i, v);
  }
}

__global__ __launch_bounds__(256) void pool2_v8(const uint16_t* __restrict__ x,
                                                int H, int W, int C, int mode,
                                                unsigned pieces,
                                                uint16_t* __restrict__ y) {
  const unsigned G = (unsigned)C / 8, Ho = (unsigned)H / 2, Wo = (unsigned)W / 2;
  const float scale = mode == 0 ? 0.25f : 1.0f;
  const int64_t rowc = (int64_t)W * C;
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < pieces; i += gridDim.x * 256) {
    const unsigned g = i % G;
    unsigned q = i / G;
    const unsigned wo = q % Wo;
    q /= Wo;
    const unsigned ho = q % Ho;
    const unsigned n = q / Ho;
    const uint16_t* b = x + ((int64_t)(n * H + 2 * ho) * W + 2 * wo) * C + 8 * g;
    float a0[8], a1[8], a2[8], a3[8], v[8];
    load8(b, a0);
    load8(b + C, a1);
    load8(b + rowc, a2);
    load8(b + rowc + C, a3);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = ((a0[k] + a1[k]) + (a2[k] + a3[k])) * scale;
    store8(y + 8 * (int64_t)i, v);
  }
}

__global__ __launch_bounds__(256) void unpool2_v8(const uint16_t* __restrict__ x,
                                                  int H, int W, int C, float scale,
                                                  unsigned pieces,
                                                  uint16_t* __restrict__ y) {
  const unsigned G = (unsigned)C / 8, Ho = 2u * H, Wo = 2u * W;
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < pieces; i += gridDim.x * 256) {
    const unsigned g = i % G;
    unsigned q = i / G;
    const unsigned wo = q % Wo;
    q /= Wo;
    const unsigned ho = q % Ho;
    const unsigned n = q / Ho;
    float v[8];
    load8(x + ((int64_t)(n * H + ho / 2) * W + wo / 2) * C + 8 * g, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] *= scale;
    store8(y + 8 * (int64_t)i, v);
  }
}

// One workgroup per sample: FP64 sum in a fixed order (strided per thread,
// then xor-shuffle and LDS across the 4 waves), then y = x - mean.
__global__ __launch_bounds__(256) void center_k(const float* x, float* y,
                                                int64_t len) {
  const float* xs = x + (int64_t)blockIdx.x * len;
  float* ys = y + (int64_t)blockIdx.x * len;
  // U loads in flight per thread before their adds, which keep the order
  // x[t], x[t + 256], x[t + 512], ... of thread t
  constexpr int U = 16;
  double s = 0.0;
  int64_t i = threadIdx.x;
  for (; i + (U - 1) * 256 < len; i += U * 256) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = xs[i + u * 256];
#pragma unroll
    for (int u = 0; u < U; ++u) s += (double)v[u];
  }
  for (; i < len; i += 256) s += (double)xs[i];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
  __shared__ double sh[4];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  const float mean = (float)(((sh[0] + sh[1]) + (sh[2] + sh[3])) / (double)len);
  // each thread reads its U values before writing them (x and y may alias)
  for (i = threadIdx.x; i + (U - 1) * 256 < len; i += U * 256) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = xs[i + u * 256];
#pragma unroll
    for (int u = 0; u < U; ++u) ys[i + u * 256] = v[u] - mean;
  }
  for (; i < len; i += 256) ys[i] = xs[i] - mean;
}

bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
  return true;
}

int grid_for(int64_t count) {
  int64_t g = (count + 255) / 256;
  return (int)(g > 65536 ? 65536 : (g < 1 ? 1 : g));
}

int launch_ok(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s launch failed: %s", what, hipGetErrorString(e));
    return SPS_E_HIP;
  }
  return SPS_OK;
}

// How each weight gradient splits its pixel reduction over workgroups; the
// workspace holds one partial gradient per workgroup (per z slice).
constexpr int64_t kPartFloats = (int64_t)16 << 20;  // partial sums, at most

struct WgradSplit {
  int blocks;    // workgroups that write a partial gradient
  int per;       // chunks (thin layers: pixels) per workgroup
  int64_t count; // floats of one partial gradient
};

// Columns of the tiled weight gradient's chunks (32, 16 or 8, the widest whose
// chunks cover the image exactly); 0 for the general kernel.  *px: pixels of a
// chunk.
int wgrad_cols(int h, int w, int cin, int cout, int* px) {
  *px = cin % 64 != 0 && cout % 64 != 0 ? 256 : 128;
  for (int wc : {32, 16, 8})
    if (w % wc == 0 && h % (*px / wc) == 0) return wc;
  *px = 32;
  return 0;
}

WgradSplit conv_split(int n, int h, int w, int cin, int cout) {
  const int kt = cout % 64 == 0 ? 64 : 32, ct = cin % 64 == 0 ? 64 : 32;
  const int64_t npix = (int64_t)n * h * w;
  const int64_t count = (int64_t)9 * cin * cout;
  const int64_t tiles = (int64_t)(cin / ct) * (cout / kt);
  int px;
  // the tiled kernel's LDS leaves one workgroup per CU: one round of 256
  const bool tiled = wgrad_cols(h, w, cin, cout, &px) != 0;
  const int64_t nchunks = npix / px;
  int64_t nz = tiled ? 256 / tiles : (2048 + tiles - 1) / tiles;
  nz = std::min<int64_t>(nz, std::max<int64_t>(1, kPartFloats / count));
  nz = std::max<int64_t>(1, std::min<int64_t>(nz, nchunks));
  const int64_t per = (nchunks + nz - 1) / nz;
  return {(int)((nchunks + per - 1) / per), (int)per, count};
}

// The thin layers: at most 1024 workgroups (four waves per SIMD) of 16 runs of
// 64 pixels at least, so that the partials stay a small share of what is read.
WgradSplit thin_split(int64_t np, int64_t count) {
  const int64_t runs = (np + 63) / 64;
  const int64_t per = std::max<int64_t>(16, (runs + 1023) / 1024);
  return {(int)((runs + per - 1) / per), (int)per * 64, count};
}

int add_parts(const float* part, const WgradSplit& sp, float* dw, hipStream_t s,
              int64_t nw = -1, float* db = nullptr) {
  if (nw < 0) nw = sp.count;
  const unsigned blocks = (unsigned)((sp.count + 63) / 64);
  if (sp.blocks > 32)
    add_partials<16><<<blocks, 1024, 0, s>>>(part, sp.blocks, sp.count, dw, nw, db);
  else
    add_partials<4><<<blocks, 256, 0, s>>>(part, sp.blocks, sp.count, dw, nw, db);
  return launch_ok("weight-gradient partial sum");
}

int check_ws(const char* who, const WgradSplit& sp, const float* ws,
             size_t ws_floats) {
  if (!ws || (int64_t)ws_floats < (int64_t)sp.blocks * sp.count) {
    set_error("%s: workspace of %zu floats is smaller than the %lld it needs "
              "(sps_nn_wgrad_workspace)", who, ws_floats,
              (long long)sp.blocks * sp.count);
    return SPS_E_INVALID;
  }
  return SPS_OK;
}

}  // namespace
}  // namespace sps

using namespace sps;

extern "C" {

int sps_nn_conv3x3(const void* x, int n, int h, int w, int cin,
                   const void* weight, const float* bias, int cout, int act,
                   int epilogue, const void* skip, void* y, void* pre,
                   void* stream) {
  const int64_t npix = (int64_t)n * h * w;
  if (!x || !weight || !y || n < 1 || h < 1 || w < 1 || cin < 32 ||
      cin % 32 || cout < 32 || cout % 32 || npix % 64 ||
      npix > (int64_t)1 << 30 || (act != 0 && act != 1) ||
      (epilogue != SPS_NN_EPI_PLAIN && epilogue != SPS_NN_EPI_UPSAMPLE_ADD) ||
      (epilogue == SPS_NN_EPI_UPSAMPLE_ADD && !skip)) {
    set_error("sps_nn_conv3x3: need cin, cout multiples of 32, n*h*w a "
              "multiple of 64, act in {0,1}, a skip tensor for UPSAMPLE_ADD");
    return SPS_E_INVALID;
  }
  hipStream_t s = (hipStream_t)stream;
  const uint16_t* xx = (const uint16_t*)x;
  const uint16_t* ww = (const uint16_t*)weight;
  const uint16_t* sk = (const uint16_t*)skip;
  uint16_t* yy = (uint16_t*)y;
  uint16_t* pp = (uint16_t*)pre;
  // LDS-tiled kernel when the image splits into whole tiles: 16 columns by
  // 8 or 16 rows, 32 / 64 / 128 output channels per workgroup
  if (w % kTileCols == 0) {
    const int tiles_w = w / kTileCols;
    // 8-wave tiles for two chunks of input channels and more (32->64 at 128^2,
    // batch 64: 90 us, conv_fwd_tile 85), where they occupy half of the 256
    // CUs at least (256->128 at 32^2 with the upsample-add epilogue,
    // batch 32, 128 workgroups: 51 us, conv_fwd_tile 78)
#define SPS_CONV_WIDE(WM, WN)                                                  \
  do {                                                                         \
    const int64_t wgs =                                                        \
        h % (4 * (WN)) || cout % (64 * (WM))                                   \
            ? 0                                                                \
            : (int64_t)n * (h / (4 * (WN))) * tiles_w * (cout / (64 * (WM)));  \
    if (cin == 32 || wgs < 128) break;                                         \
    if (epilogue == SPS_NN_EPI_PLAIN)                                          \
      conv_fwd_wide<WM, WN, 0><<<(unsigned)wgs, 512, 0, s>>>(                  \
          xx, h, w, cin, ww, bias, cout, act, sk, yy, pp);                     \
    else                                                                       \
      conv_fwd_wide<WM, WN, 1><<<(unsigned)wgs, 512, 0, s>>>(                  \
          xx, h, w, cin, ww, bias, cout, act, sk, yy, pp);                     \
    return launch_ok("sps_nn_conv3x3");                                        \
  } while (0)
    SPS_CONV_WIDE(2, 4);
    SPS_CONV_WIDE(1, 8);
#undef SPS_CONV_WIDE
#define SPS_CONV_TILE(MW, NW, WM, WN)                                           \
  do {                                                                         \
    constexpr int TH_ = (NW) * (WN), KB_ = 16 * (MW) * (WM);                   \
    /* two chunks staged at once only where registers allow 3 waves/SIMD */   \
    constexpr int C2_ = (MW) == 2 ? 2 : 0;                                     \
    dim3 g((unsigned)(n * (h / TH_) * tiles_w), (unsigned)(cout / KB_));      \
    if (epilogue == SPS_NN_EPI_PLAIN && cin == 32)                             \
      conv_fwd_tile<MW, NW, WM, WN, 0, 1><<<g, 256, 0, s>>>(                    \
          xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp);                  \
    else if (epilogue == SPS_NN_EPI_PLAIN && cin == 64 && C2_)                 \
      conv_fwd_tile<MW, NW, WM, WN, 0, C2_><<<g, 256, 0, s>>>(                  \
          xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp);                  \
    else if (epilogue == SPS_NN_EPI_PLAIN)                                     \
      conv_fwd_tile<MW, NW, WM, WN, 0, 0><<<g, 256, 0, s>>>(                    \
          xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp);                  \
    else if (cin == 64 && C2_)                                                 \
      conv_fwd_tile<MW, NW, WM, WN, 1, C2_><<<g, 256, 0, s>>>(                  \
          xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp);                  \
    else                                                                       \
      conv_fwd_tile<MW, NW, WM, WN, 1, 0><<<g, 256, 0, s>>>(                    \
          xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp);                  \
    return launch_ok("sps_nn_conv3x3");                                        \
  } while (0)
    // the upsample-add epilogue stages through LDS: 64 channels x 8 rows
    if (epilogue == SPS_NN_EPI_UPSAMPLE_ADD && cout % 64 == 0 && h % 8 == 0)
      SPS_CONV_TILE(4, 2, 1, 4);
    if (cout % 128 == 0 && h % 8 == 0) SPS_CONV_TILE(4, 4, 2, 2);
    if (cout % 64 == 0 && h % 16 == 0) SPS_CONV_TILE(4, 4, 1, 4);
    if (cout % 64 == 0 && h % 8 == 0) SPS_CONV_TILE(4, 2, 1, 4);
    if (h % 16 == 0) SPS_CONV_TILE(2, 4, 1, 4);
    if (h % 8 == 0) SPS_CONV_TILE(2, 2, 1, 4);
#undef SPS_CONV_TILE
  }
  const int nt = cout % 64 == 0 ? 4 : 2;
  dim3 grid((unsigned)((npix / 64 + 3) / 4), (unsigned)(cout / (16 * nt)));
  if (epilogue == SPS_NN_EPI_PLAIN) {
    if (nt == 4)
      conv_fwd<4, 0><<<grid, 256, 0, s>>>(xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp, (int)npix);
    else
      conv_fwd<2, 0><<<grid, 256, 0, s>>>(xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp, (int)npix);
  } else {
    if (nt == 4)
      conv_fwd<4, 1><<<grid, 256, 0, s>>>(xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp, (int)npix);
    else
      conv_fwd<2, 1><<<grid, 256, 0, s>>>(xx, n, h, w, cin, ww, bias, cout, act, sk, yy, pp, (int)npix);
  }
  return launch_ok("sps_nn_conv3x3");
}

size_t sps_nn_wgrad_workspace(int kind, int n, int h, int w, int cin,
                              int cout) {
  if (n < 1 || h < 1 || w < 1 || cin < 1 || cout < 1) return 0;
  const int64_t np = (int64_t)n * h * w;
  WgradSplit sp{0, 0, 0};
  if (kind == SPS_NN_WGRAD_CONV) {
    sp = conv_split(n, h, w, cin, cout);
    sp.count += cout;  // the bias gradient
  } else if (kind == SPS_NN_WGRAD_IN1) sp = thin_split(np, (int64_t)10 * cout);
  else if (kind == SPS_NN_WGRAD_OUT1) sp = thin_split(np, (int64_t)9 * cin);
  return (size_t)((int64_t)sp.blocks * sp.count);
}

int sps_nn_conv3x3_wgrad(const void* x, const void* dpre, int n, int h, int w,
                         int cin, int cout, float* dweight, float* workspace,
                         size_t ws_floats, void* stream) {
  return sps_nn_conv3x3_wgrad_bias(x, dpre, n, h, w, cin, cout, dweight, nullptr,
                                   workspace, ws_floats, stream);
}

int sps_nn_conv3x3_wgrad_bias(const void* x, const void* dpre, int n, int h,
                              int w, int cin, int cout, float* dweight,
                              float* dbias, float* workspace, size_t ws_floats,
                              void* stream) {
  const int64_t npix = (int64_t)n * h * w;
  if (!x || !dpre || !dweight || n < 1 || h < 1 || w < 1 || npix % 32 ||
      npix > (int64_t)1 << 30 || cin % 32 || cout % 32 || cin < 32 ||
      cout < 32) {
    set_error("sps_nn_conv3x3_wgrad: need n*h*w, cin, cout multiples of 32");
    return SPS_E_INVALID;
  }
  WgradSplit sp = conv_split(n, h, w, cin, cout);
  const int64_t nw = sp.count;
  if (dbias) sp.count += cout;
  SPS_TRY(check_ws("sps_nn_conv3x3_wgrad", sp, workspace, ws_floats));
  int px;
  const int wc = wgrad_cols(h, w, cin, cout, &px);
  const int nchunks = (int)(npix / px);
  const int per = sp.per;
  const int kt = cout % 64 == 0 ? 64 : 32;
  const int ct = cin % 64 == 0 ? 64 : 32;
  dim3 grid(cin / ct, cout / kt, sp.blocks);
  hipStream_t s = (hipStream_t)stream;
  const uint16_t* xx = (const uint16_t*)x;
  const uint16_t* dd = (const uint16_t*)dpre;
#define SPS_WGRAD_TILE(KT_, CT_, WC_)                                         \
  conv_wgrad_tile<KT_, CT_, WC_><<<grid, 512, 0, s>>>(                        \
      xx, dd, h, w, cin, cout, workspace, sp.count, nchunks, per, dbias != nullptr)
#define SPS_WGRAD(KT_, CT_)                                                   \
  do {                                                                        \
    if (wc == 32) SPS_WGRAD_TILE(KT_, CT_, 32);                               \
    else if (wc == 16) SPS_WGRAD_TILE(KT_, CT_, 16);                          \
    else if (wc == 8) SPS_WGRAD_TILE(KT_, CT_, 8);                            \
    else if (w % 32 == 0)                                                     \
      conv_wgrad<KT_, CT_, true><<<grid, 256, 0, s>>>(                        \
          xx, dd, n, h, w, cin, cout, workspace, sp.count, nchunks, per,      \
          dbias != nullptr);                                                  \
    else                                                                      \
      conv_wgrad<KT_, CT_, false><<<grid, 256, 0, s>>>(                       \
          xx, dd, n, h, w, cin, cout, workspace, sp.count, nchunks, per,      \
          dbias != nullptr);                                                  \
  } while (0)
  if (kt == 64 && ct == 64)
    SPS_WGRAD(64, 64);
  else if (kt == 64)
    SPS_WGRAD(64, 32);
  else if (ct == 64)
    SPS_WGRAD(32, 64);
  else
    SPS_WGRAD(32, 32);
#undef SPS_WGRAD
#undef SPS_WGRAD_TILE
  SPS_TRY(launch_ok("sps_nn_conv3x3_wgrad"));
  return add_parts(workspace, sp, dweight, s, nw, dbias);
}

int sps_nn_conv3x3_in1(const float* x, int n, int h, int w,
                       const float* weight, const float* bias, int cout,
                       int act, void* y, void* pre, void* stream) {
  const int64_t np = (int64_t)n * h * w;
  if (!x || !weight || !y || np < 1 || cout < 8 || cout > 64 || cout % 8 ||
      (act != 0 && act != 1)) {
    set_error("sps_nn_conv3x3_in1: cout a multiple of 8 in 8..64, act 0/1");
    return SPS_E_INVALID;
  }
  const unsigned blocks = (unsigned)((np + 255) / 256);
  if (cout == 32)
    in1_fwd_staged<32><<<blocks, 256, 0, (hipStream_t)stream>>>(
        x, n, h, w, weight, bias, act, (uint16_t*)y, (uint16_t*)pre);
  else if (cout == 64)
    in1_fwd_staged<64><<<blocks, 256, 0, (hipStream_t)stream>>>(
        x, n, h, w, weight, bias, act, (uint16_t*)y, (uint16_t*)pre);
  else
    in1_fwd<<<blocks, 256, 0, (hipStream_t)stream>>>(
        x, n, h, w, weight, bias, cout, act, (uint16_t*)y, (uint16_t*)pre);
  return launch_ok("sps_nn_conv3x3_in1");
}

int sps_nn_conv3x3_in1_wgrad(const float* x, const void* dpre, int n, int h,
                             int w, int cout, float* dweight, float* workspace,
                             size_t ws_floats, void* stream) {
  return sps_nn_conv3x3_in1_wgrad_bias(x, dpre, n, h, w, cout, dweight, nullptr,
                                       workspace, ws_floats, stream);
}

int sps_nn_conv3x3_in1_wgrad_bias(const float* x, const void* dpre, int n,
                                  int h, int w, int cout, float* dweight,
                                  float* dbias, float* workspace,
                                  size_t ws_floats, void* stream) {
  const int64_t np = (int64_t)n * h * w;
  if (!x || !dpre || !dweight || np < 1 || cout < 8 || cout > 64 || cout % 8) {
    set_error("sps_nn_conv3x3_in1_wgrad: cout a multiple of 8 in 8..64");
    return SPS_E_INVALID;
  }
  const WgradSplit sp = thin_split(np, (int64_t)(dbias ? 10 : 9) * cout);
  SPS_TRY(check_ws("sps_nn_conv3x3_in1_wgrad", sp, workspace, ws_floats));
  hipStream_t s = (hipStream_t)stream;
  thin_wgrad<1><<<dim3((unsigned)sp.blocks, (cout + 31) / 32), 256, 0, s>>>(
      (const uint16_t*)dpre, x, np, h, w, cout, workspace, sp.count, sp.per,
      dbias != nullptr);
  SPS_TRY(launch_ok("sps_nn_conv3x3_in1_wgrad"));
  return add_parts(workspace, sp, dweight, s, (int64_t)9 * cout, dbias);
}

int sps_nn_conv3x3_out1(const void* x, int n, int h, int w, int cin,
                        const float* weight, const float* bias, float* y,
                        void* stream) {
  const int64_t np = (int64_t)n * h * w;
  if (!x || !weight || !y || np < 1 || cin < 8 || cin > 64 || cin % 8) {
    set_error("sps_nn_conv3x3_out1: cin a multiple of 8 in 8..64");
    return SPS_E_INVALID;
  }
  const unsigned tiles = (unsigned)(n * (h / 16) * (w / 16));
  if (h % 16 == 0 && w % 16 == 0 && cin == 32)
    out1_fwd_tile<32><<<tiles, 256, 0, (hipStream_t)stream>>>(
        (const uint16_t*)x, n, h, w, weight, bias, y);
  else if (h % 16 == 0 && w % 16 == 0 && cin == 64)
    out1_fwd_tile<64><<<tiles, 256, 0, (hipStream_t)stream>>>(
        (const uint16_t*)x, n, h, w, weight, bias, y);
  else
    out1_fwd<<<(unsigned)((np + 255) / 256), 256, 0, (hipStream_t)stream>>>(
        (const uint16_t*)x, n, h, w, cin, weight, bias, y);
  return launch_ok("sps_nn_conv3x3_out1");
}

int sps_nn_conv3x3_out1_bwd(const void* x, const float* dy, int n, int h,
                            int w, int cin, const float* weight, void* dx,
                            float* dweight, float* workspace, size_t ws_floats,
                            void* stream) {
  const int64_t np = (int64_t)n * h * w;
  if (!x || !dy || !weight || np < 1 || cin < 8 || cin > 64 || cin % 8) {
    set_error("sps_nn_conv3x3_out1_bwd: cin a multiple of 8 in 8..64");
    return SPS_E_INVALID;
  }
  hipStream_t s = (hipStream_t)stream;
  const WgradSplit sp = thin_split(np, (int64_t)9 * cin);
  if (dweight) SPS_TRY(check_ws("sps_nn_conv3x3_out1_bwd", sp, workspace, ws_floats));
  if (dx) {
    out1_bwd_data<<<(unsigned)((np + 255) / 256), 256, 0, s>>>(
        dy, n, h, w, cin, weight, (uint16_t*)dx);
    SPS_TRY(launch_ok("sps_nn_conv3x3_out1_bwd (data)"));
  }
  if (dweight) {
    thin_wgrad<-1><<<dim3((unsigned)sp.blocks, (cin + 31) / 32), 256, 0, s>>>(
        (const uint16_t*)x, dy, np, h, w, cin, workspace, sp.count, sp.per, 0);
    SPS_TRY(launch_ok("sps_nn_conv3x3_out1_bwd (weight)"));
    SPS_TRY(add_parts(workspace, sp, dweight, s));
  }
  return SPS_OK;
}

int sps_nn_silu_bwd(const void* dy, const void* pre, void* dx, size_t count,
                    void* stream) {
  if (!dy || !pre || !dx) {
    set_error("sps_nn_silu_bwd: NULL pointer");
    return SPS_E_INVALID;
  }
  if (count % 8 == 0 && count / 8 < ((size_t)1 << 31) &&
      aligned16({dy, pre, dx})) {
    silu_bwd_v8<<<grid_for((int64_t)(count / 8)), 256, 0, (hipStream_t)stream>>>(
        (const uint16_t*)dy, (const uint16_t*)pre, (uint16_t*)dx, (unsigned)(count / 8));
    return launch_ok("sps_nn_silu_bwd");
  }
  silu_bwd_k<<<grid_for((int64_t)count), 256, 0, (hipStream_t)stream>>>(
      (const uint16_t*)dy, (const uint16_t*)pre, (uint16_t*)dx, (int64_t)count);
  return launch_ok("sps_nn_silu_bwd");
}

int sps_nn_pool2(const void* x, int n, int h, int w, int c, int mode, void* y,
                 void* stream) {
  if (!x || !y || h % 2 || w % 2 || c < 1 || (mode != 0 && mode != 1)) {
    set_error("sps_nn_pool2: even h and w, mode 0 or 1");
    return SPS_E_INVALID;
  }
  const int64_t pieces = (int64_t)n * (h / 2) * (w / 2) * (c / 8);
  if (c % 8 == 0 && pieces < ((int64_t)1 << 31) && aligned16({x, y})) {
    pool2_v8<<<grid_for(pieces), 256, 0, (hipStream_t)stream>>>(
        (const uint16_t*)x, h, w, c, mode, (unsigned)pieces, (uint16_t*)y);
    return launch_ok("sps_nn_pool2");
  }
  pool2_k<<<grid_for((int64_t)n * h * w * c / 4), 256, 0, (hipStream_t)stream>>>(
      (const uint16_t*)x, n, h, w, c, mode, (uint16_t*)y);
  return launch_ok("sps_nn_pool2");
}

int sps_nn_center(const float* x, float* y, int n, int64_t len,
                  void* stream) {
  if (!x || !y || n < 1 || len < 1) {
    set_error("sps_nn_center: NULL pointer or empty samples");
    return SPS_E_INVALID;
  }
  center_k<<<(unsigned)n, 256, 0, (hipStream_t)stream>>>(x, y, len);
  return launch_ok("sps_nn_center");
}

int sps_nn_unpool2(const void* x, int n, int h, int w, int c, float scale,
                   void* y, void* stream) {
  if (!x || !y || c < 1) {
    set_error("sps_nn_unpool2: invalid arguments");
    return SPS_E_INVALID;
  }
  const int64_t pieces = (int64_t)n * (2 * h) * (2 * w) * (c / 8);
  if (c % 8 == 0 && pieces < ((int64_t)1 << 31) && aligned16({x, y})) {
    unpool2_v8<<<grid_for(pieces), 256, 0, (hipStream_t)stream>>>(
        (const uint16_t*)x, h, w, c, scale, (unsigned)pieces, (uint16_t*)y);
    return launch_ok("sps_nn_unpool2");
  }
  unpool2_k<<<grid_for((int64_t)n * h * w * c * 4), 256, 0, (hipStream_t)stream>>>(
      (const uint16_t*)x, n, h, w, c, scale, (uint16_t*)y);
  return launch_ok("sps_nn_unpool2");
}

}  // extern "C"
