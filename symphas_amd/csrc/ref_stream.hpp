// ref_stream.hpp - the reference-order step of a periodic field (or two
// coupled ones) as a stream of rows (2D) or planes (3D).
//
// Same arithmetic as the one-site-per-thread kernels, value for value and in
// the same order (stencil_ref.hpp's groupings, terms in descriptor order, no
// FMA: include it only in files compiled with -ffp-contract=off), so the bits
// are theirs; what changes is where the operands come from:
//   - a wave owns 60 columns (64 lanes, two halo lanes per side) and streams
//     the rows of a chunk; a site is loaded once per chunk instead of once per
//     stencil point, x neighbours come from adjacent lanes (DPP) and y
//     neighbours from the rows held in registers;
//   - the operand of a laplacian of a polynomial (or monomial) is evaluated
//     once per site, as the reference's temporary grid is, instead of at every
//     stencil point;
//   - which derivatives a step takes is known at compile time.
// The one-site kernel interprets the term list: 290 VALU and 24 loads per site
// of Model B, bound by issue.  The stream takes about 75 (50 of them the FP64
// adds and products that the order asks for) and one load, and is bound by the
// latency of those sums on small fields and by issue on large ones.
// Model B <9,6,13> FP64 1023x769: 25.9 -> 6.6 us per step; Model C <9,6,13>
// FP64 641x450: 211 -> 5.4 us.
#pragma once

#include "common.hpp"
#include "fused_tile.hpp"
#include "lanes.hpp"
#include "shape.hpp"
#include "stencil_ref.hpp"

namespace sps {

// rows of one operand: centre value and its x neighbours, slot = row mod 5
template <typename T>
struct RsWindow {
  T m[5], c[5], p[5];
  __device__ __forceinline__ void push(int slot, T v) {
    c[slot] = v;
    m[slot] = from_prev_lane(v);
    p[slot] = from_next_lane(v);
  }
};

// stencil accessor on a window whose newest row (slot PH) is two rows above
// the output row
template <typename T, int PH>
struct RsAcc {
  const RsWindow<T>* w;
  __device__ __forceinline__ T operator()(int i, int j, int) const {
    const int s = (PH + 3 + j) % 5;
    switch (i) {
      case -2: return from_prev_lane(w->m[s]);
      case -1: return w->m[s];
      case 0: return w->c[s];
      case 1: return w->p[s];
      default: return from_next_lane(w->p[s]);
    }
  }
};

// the laplacian and bilaplacian of a point count (5, 9: 2D, the others 3D)
template <int L, typename T, class A>
__device__ __forceinline__ T rs_lap(const A& a, T divh2) {
  if constexpr (L == 5)
    return ref::lap2_5<T>(a, divh2);
  else if constexpr (L == 9)
    return ref::lap2_9<T>(a, divh2);
  else if constexpr (L == 7)
    return ref::lap3_7<T>(a, divh2);
  else
    return ref::lap3_15<T>(a, divh2);
}

template <int B, typename T, class A>
__device__ __forceinline__ T rs_bilap(const A& a, T divh4) {
  if constexpr (B == 13)
    return ref::bilap2_13<T>(a, divh4);
  else if constexpr (B == 17)
    return ref::bilap2_17<T>(a, divh4);
  else if constexpr (B == 21)
    return ref::bilap2_21<T>(a, divh4);
  else
    return ref::bilap3_25<T>(a, divh4);
}

template <typename T, int NF>
struct RsFields {
  const T* in[NF];
  T* out[NF];
  int X, Y, Z, TY, TZ, nstrips, nrowblk, nitems;  // Z, TZ, nrowblk: 3D
};

// Prog supplies the model:
//   NF fields, NLAP operands under a laplacian that are not a field;
//   lap_operand<d>(x): such an operand at a site with field values x;
//   rhs(F, D, x, r): the right-hand sides r at a site with field values x,
//   from stencil accessors F of the fields and D of the operands.
template <typename T, class Prog>
__global__ __launch_bounds__(64) void ref_stream2d(
    const RsFields<T, Prog::NF> g, const Prog p) {
  constexpr int NF = Prog::NF, NLAP = Prog::NLAP;
  constexpr int W = 60;
  const int lane = threadIdx.x;
  const int item =
      __builtin_amdgcn_readfirstlane(xcd_remap(blockIdx.x, gridDim.x));
  if (item >= g.nitems) return;
  const int strip = item % g.nstrips, chunk = item / g.nstrips;
  const int X = g.X, Y = g.Y;
  const int cb = strip * W + lane - 2;
  int col = cb % X;
  if (col < 0) col += X;
  const bool store_lane = lane >= 2 && lane < 62 && cb < X;
  const int y0 = chunk * g.TY;
  const int ty = min(g.TY, Y - y0);
  const int NI = ty + 4;
  int rload = (y0 - 2) % Y;
  if (rload < 0) rload += Y;

  // a wave-uniform descriptor per row; lanes that do not store get an offset
  // past the row, whose stores the range check drops
  const int row_bytes = X * (int)sizeof(T);
  const unsigned ld_off = (unsigned)col * (unsigned)sizeof(T);
  const unsigned st_off = store_lane ? ld_off : 0x80000000u;
  T ring[5][NF];
  auto load_row = [&](T (&b)[NF]) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      T v[1];
      buf_load<T, 1>(buffer_rsrc(g.in[f] + (int64_t)rload * X, row_bytes),
                     ld_off, 0, v);
      b[f] = v[0];
    }
    rload = rload + 1 == Y ? 0 : rload + 1;
  };
  static_for<0, 5>([&](auto u) { load_row(ring[decltype(u)::value]); });

  RsWindow<T> F[NF];
  RsWindow<T> D[NLAP > 0 ? NLAP : 1];
  int64_t orow = (int64_t)y0 * X;

  auto take = [&](auto ic) {
    constexpr int S = decltype(ic)::value % 5;
    T x[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      x[f] = ring[S][f];
      F[f].push(S, x[f]);
    }
    static_for<0, NLAP>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      D[d].push(S, p.template lap_operand<d>(x));
    });
    load_row(ring[S]);
  };
  auto emit = [&](auto ic) {
    constexpr int S = decltype(ic)::value % 5;
    T x[NF], r[NF];
    RsAcc<T, S> a[NF], d[NLAP > 0 ? NLAP : 1];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      x[f] = F[f].c[(S + 3) % 5];
      a[f].w = &F[f];
    }
#pragma unroll
    for (int q = 0; q < NLAP; ++q) d[q].w = &D[q];
    p.rhs(a, d, x, r);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      // forward Euler psi + dt*dframe (examples/solvers/solverft.h:46-50)
      T v[1] = {x[f] + p.dt * r[f]};
      buf_store<T, 1>(buffer_rsrc(g.out[f] + orow, row_bytes), st_off, 0, v);
    }
    orow += X;
  };

  static_for<0, 4>([&](auto u) { take(u); });
  int i = 4;
  for (; i + 5 <= NI; i += 5)
    static_for<0, 5>([&](auto u) {
      take(std::integral_constant<int, 4 + decltype(u)::value>{});
      emit(std::integral_constant<int, 4 + decltype(u)::value>{});
    });
  static_for<0, 4>([&](auto u) {
    if (i + decltype(u)::value < NI) {
      take(std::integral_constant<int, 4 + decltype(u)::value>{});
      emit(std::integral_constant<int, 4 + decltype(u)::value>{});
    }
  });
}

// Chunk height.  A row costs about 0.3 us in a lone wave (the stencils' sums
// are serial) and a chunk streams 4 fill rows, so small fields take the lowest
// chunks and large ones grow them once six waves per SIMD of the 1024 are
// busy.  Model B <9,6,13> FP64, us per step at 4 / 16 / 32 / 64 rows: 257x301
// 4.2 / 7.3 / 11.4 / 19.9; 1023x769 6.6 / 8.6 / 12.6 / 20.6; 4096x4096 62.1 /
// 53.3 / 53.1 / 55.2.
inline int ref_stream_rows(int Y, int nstrips) {
  constexpr int64_t kWaves = 6 * 1024;
  const int64_t ty = ((int64_t)Y * nstrips + kWaves - 1) / kWaves;
  return (int)(ty < 4 ? 4 : (ty > 32 ? 32 : ty));
}

template <typename T, class Prog>
void launch_ref_stream2d(RsFields<T, Prog::NF> g, const Prog& p,
                         hipStream_t s) {
  g.nstrips = (g.X + 59) / 60;
  g.TY = ref_stream_rows(g.Y, g.nstrips);
  g.nitems = g.nstrips * ((g.Y + g.TY - 1) / g.TY);
  ref_stream2d<T, Prog><<<g.nitems, 64, 0, s>>>(g, p);
}

// ---------------------------------------------------------------------- 3D

// stencil accessor on planes (slot = plane mod 5, the newest in slot PH two
// planes above the output) of rows r - 2 .. of the wave's columns
template <typename T, int PH, int NP>
struct RsAcc3 {
  const T (*w)[NP];  // [slot][row]
  int r;             // the output row's index in a plane
  __device__ __forceinline__ T operator()(int i, int j, int k) const {
    const T c = w[(PH + 3 + k) % 5][r + j];
    switch (i) {
      case -2: return from_prev_lane(from_prev_lane(c));
      case -1: return from_prev_lane(c);
      case 0: return c;
      case 1: return from_next_lane(c);
      default: return from_next_lane(from_next_lane(c));
    }
  }
};

// One wave owns 60 columns x TYW rows and streams the planes of a z-chunk, as
// the fused 3D stream does; the five planes in reach stay in registers and x
// neighbours come through DPP.  The one-site kernel reads 15 to 25 neighbours
// per derivative and evaluates an operand at each of them.
// Bound by issue and the sums' latency.  <15,10,25>, us per step: Model B FP64
// 161x150x97 272 -> 24, FP32 256^3 699 -> 74; Model C FP64 161x150x97 2380 ->
// 44.
template <typename T, int TYW, class Prog>
__global__ __launch_bounds__(256) void ref_stream3d(
    const RsFields<T, Prog::NF> g, const Prog p) {
  constexpr int NF = Prog::NF, NLAP = Prog::NLAP;
  constexpr int W = 60, NP = TYW + 4;
  const int lane = threadIdx.x & 63;
  const int item = __builtin_amdgcn_readfirstlane(
      xcd_remap(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6));
  if (item >= g.nitems) return;
  const int X = g.X, Y = g.Y, Z = g.Z;
  const int strip = item % g.nstrips;
  const int rb = (item / g.nstrips) % g.nrowblk;
  const int zc = item / (g.nstrips * g.nrowblk);
  const int x0 = strip * W + lane - 2;
  int col = x0 % X;
  if (col < 0) col += X;
  const bool store_lane = lane >= 2 && lane < 62 && x0 < X;
  const int y0 = rb * TYW, z0 = zc * g.TZ;
  const int NI = min(g.TZ, Z - z0) + 4;
  const int64_t XY = (int64_t)X * Y;
  int rowoff[NP];
#pragma unroll
  for (int r = 0; r < NP; ++r) {
    int y = (y0 - 2 + r) % Y;
    if (y < 0) y += Y;
    rowoff[r] = __builtin_amdgcn_readfirstlane(y * X);
  }
  int zl = (z0 - 2) % Z;
  if (zl < 0) zl += Z;

  T F[NF][5][NP], D[NLAP > 0 ? NLAP : 1][5][NP];
  T NX[NF][NP];
  auto fetch = [&]() {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int r = 0; r < NP; ++r)
        NX[f][r] = (g.in[f] + (int64_t)zl * XY + rowoff[r])[col];
    zl = zl + 1 == Z ? 0 : zl + 1;
  };
  fetch();
  for (int i = 0; i < NI; i += 5)
    static_for<0, 5>([&](auto uc) {
      constexpr int S = decltype(uc)::value;
      if (i + S < NI) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int r = 0; r < NP; ++r) F[f][S][r] = NX[f][r];
        if (i + S + 1 < NI) fetch();
        // operands: laplacians reach one row
#pragma unroll
        for (int r = 1; r < NP - 1; ++r) {
          T x[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) x[f] = F[f][S][r];
          static_for<0, NLAP>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            D[d][S][r] = p.template lap_operand<d>(x);
          });
        }
        if (i + S >= 4) {
          T v[NF][TYW];
#pragma unroll
          for (int r = 0; r < TYW; ++r) {
            T x[NF], rr[NF];
            RsAcc3<T, S, NP> a[NF], d[NLAP > 0 ? NLAP : 1];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              x[f] = F[f][(S + 3) % 5][r + 2];
              a[f].w = F[f];
              a[f].r = r + 2;
            }
#pragma unroll
            for (int q = 0; q < NLAP; ++q) {
              d[q].w = D[q];
              d[q].r = r + 2;
            }
            p.rhs(a, d, x, rr);
#pragma unroll
            for (int f = 0; f < NF; ++f) v[f][r] = x[f] + p.dt * rr[f];
          }
          if (store_lane) {
            const int64_t o = (int64_t)(z0 + i + S - 4) * XY + col;
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
              for (int r = 0; r < TYW; ++r)
                if (y0 + r < Y) g.out[f][o + rowoff[r + 2]] = v[f][r];
          }
        }
      }
    });
}

// Chunk heights from the cost of shape.hpp over a few (a plane in a lone wave
// costs 1.3 of a shared one).
template <typename T, int TYW, class Prog>
void launch_ref_stream3d(RsFields<T, Prog::NF> g, const Prog& p,
                         hipStream_t s) {
  g.nstrips = (g.X + 59) / 60;
  g.nrowblk = (g.Y + TYW - 1) / TYW;
  const int64_t per_chunk = (int64_t)g.nstrips * g.nrowblk;
  double least = 0;
  for (int tz : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 256, 1024}) {
    const int64_t waves = per_chunk * ((g.Z + tz - 1) / tz);
    const double cost =
        (tz + 4) * std::max(1.3, (double)((waves + kSimds - 1) / kSimds));
    if (least == 0 || cost < least) {
      least = cost;
      g.TZ = tz;
    }
  }
  g.nitems = (int)(per_chunk * ((g.Z + g.TZ - 1) / g.TZ));
  ref_stream3d<T, TYW, Prog>
      <<<(unsigned)(((int64_t)g.nitems + 3) / 4), 256, 0, s>>>(g, p);
}

}  // namespace sps
