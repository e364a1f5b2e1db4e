// ref_stream.hpp - the reference-order step of a 2D periodic field (or two
// coupled ones) as a row stream.
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
  const RsWindow<T>& w;
  __device__ __forceinline__ T operator()(int i, int j, int) const {
    const int s = (PH + 3 + j) % 5;
    switch (i) {
      case -2: return from_prev_lane(w.m[s]);
      case -1: return w.m[s];
      case 0: return w.c[s];
      case 1: return w.p[s];
      default: return from_next_lane(w.p[s]);
    }
  }
};

template <typename T, int L, class A>
__device__ __forceinline__ T rs_lap2(const A& a, T divh2) {
  if constexpr (L == 5)
    return ref::lap2_5<T>(a, divh2);
  else
    return ref::lap2_9<T>(a, divh2);
}

template <typename T, int B, class A>
__device__ __forceinline__ T rs_bilap2(const A& a, T divh4) {
  if constexpr (B == 13)
    return ref::bilap2_13<T>(a, divh4);
  else if constexpr (B == 17)
    return ref::bilap2_17<T>(a, divh4);
  else
    return ref::bilap2_21<T>(a, divh4);
}

template <typename T, int NF>
struct RsFields {
  const T* in[NF];
  T* out[NF];
  int X, Y, TY, nstrips, nitems;
};

// Prog supplies the model:
//   NF fields, NLAP operands under a laplacian that are not a field;
//   lap_operand<d>(x): such an operand at a site with field values x;
//   rhs<S>(F, D, x, r): the right-hand sides from the fields' windows F and
//   the operands' windows D, whose newest row is in slot S.
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
#pragma unroll
    for (int f = 0; f < NF; ++f) x[f] = F[f].c[(S + 3) % 5];
    p.template rhs<S>(F, D, x, r);
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

}  // namespace sps
