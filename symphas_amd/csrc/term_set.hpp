// term_set.hpp - a right-hand side as a set of kinds of terms, for the
// reference-order streams (ref_stream.hpp; same compile flags).
#pragma once

#include <cstring>

#include "ref_stream.hpp"

namespace sps {

// A right-hand side of up to three terms, each of another kind of these four:
enum { kSLap = 1, kSLapOp = 2, kSBilap = 4, kSId = 8 };
// the laplacian of psi, the laplacian of a polynomial of psi, the bilaplacian
// of psi, a polynomial of psi.

// sum_k c[k] x^k in increasing degree, x^k as a product of k copies, zero
// coefficients skipped (mask has bit k set where c[k] != 0): poly_eval with
// its common forms first
template <typename T>
struct PolyOperand {
  T c[kMaxDeg + 1];
  int mask;
  __device__ __forceinline__ T eval(T x) const {
    const T x2 = x * x, x3 = x2 * x;
    if (mask == 8) return c[3] * x3;
    if (mask == 10) return c[1] * x + c[3] * x3;
    T acc = T(0), pw = x;
#pragma unroll
    for (int k = 0; k <= kMaxDeg; ++k) {
      if (k >= 2) pw = pw * x;
      if ((mask >> k) & 1) {
        const T t = k == 0 ? c[0] : c[k] * pw;
        acc = (mask & ((1 << k) - 1)) ? acc + t : t;
      }
    }
    return acc;
  }
};

template <typename T, int SET, int L, int B>
struct TermSet {
  static constexpr int NF = 1;
  static constexpr int NLAP = (SET & kSLapOp) ? 1 : 0;
  static constexpr int N = __builtin_popcount(SET);
  T coeff[4];  // of each kind, in the order of the bits
  // of three terms, the one summed last (as an index of the set's members);
  // the first two commute
  int last;
  PolyOperand<T> lap_op, id_op;
  T divh2, divh4, dt;

  template <int d>
  __device__ __forceinline__ T lap_operand(const T (&x)[1]) const {
    return lap_op.eval(x[0]);
  }
  template <class A>
  __device__ __forceinline__ void rhs(const A (&a)[1], const A (&d)[1],
                                      const T (&x)[1], T (&r)[1]) const {
    T v[N];
    int n = 0;
    if constexpr (SET & kSLap) v[n++] = coeff[0] * rs_lap<L>(a[0], divh2);
    if constexpr (SET & kSLapOp) v[n++] = coeff[1] * rs_lap<L>(d[0], divh2);
    if constexpr (SET & kSBilap) v[n++] = coeff[2] * rs_bilap<B>(a[0], divh4);
    if constexpr (SET & kSId) v[n++] = coeff[3] * id_op.eval(x[0]);
    if constexpr (N == 1) {
      r[0] = v[0];
    } else if constexpr (N == 2) {
      r[0] = v[0] + v[1];
    } else {
      if (last == 2) r[0] = (v[0] + v[1]) + v[2];
      else if (last == 1) r[0] = (v[0] + v[2]) + v[1];
      else r[0] = (v[1] + v[2]) + v[0];
    }
  }
};

// Which kind each term is; 0 when the list is not a set of the above: a
// gradlaplacian, a provisional variable, a bilaplacian of other than psi, two
// terms of a kind, more than three terms or none.
template <typename T>
int term_set(const RefParams<T>& p, int (&kind)[3]) {
  if (p.mode != 0 || p.nterms < 1 || p.nterms > 3) return 0;
  int set = 0;
  for (int t = 0; t < p.nterms; ++t) {
    const DevTerm<T>& tm = p.terms[t];
    if (tm.operand != 0) return 0;
    kind[t] = tm.op == SPS_OP_ID    ? kSId
              : tm.op == SPS_OP_LAP ? (tm.identity ? kSLap : kSLapOp)
              : tm.op == SPS_OP_BILAP && tm.identity ? kSBilap : 0;
    if (kind[t] == 0 || (set & kind[t])) return 0;
    set |= kind[t];
  }
  return set;
}

// The set's parameters from the step's.
template <typename T, int SET, int L, int B>
TermSet<T, SET, L, B> make_term_set(const RefParams<T>& p, const int (&kind)[3]) {
  TermSet<T, SET, L, B> ts;
  std::memset(&ts, 0, sizeof(ts));
  for (int t = 0; t < p.nterms; ++t) {
    const DevTerm<T>& tm = p.terms[t];
    ts.coeff[__builtin_ctz(kind[t])] = tm.coeff;
    ts.last = __builtin_popcount(SET & (kind[t] - 1));
    if (kind[t] == kSLapOp || kind[t] == kSId) {
      PolyOperand<T>& o = kind[t] == kSId ? ts.id_op : ts.lap_op;
      for (int k = 0; k <= kMaxDeg; ++k) {
        o.c[k] = tm.poly[k];
        if (tm.poly[k] != T(0)) o.mask |= 1 << k;
      }
    }
  }
  ts.divh2 = p.divh2;
  ts.divh4 = p.divh4;
  ts.dt = p.dt;
  return ts;
}

template <typename T>
RsFields<T, 1> stream_fields(const T* in, T* out, const RefParams<T>& p) {
  RsFields<T, 1> g;
  std::memset(&g, 0, sizeof(g));
  g.in[0] = in;
  g.out[0] = out;
  g.X = p.n[0];
  g.Y = p.n[1];
  g.Z = p.n[2];
  return g;
}

// Launches the step of a 3D set, when one of the 3D streams takes it (false:
// no stream of that set and stencils).
template <typename T>
bool launch_ref_set3d(int set, const T* in, T* out, const RefParams<T>& p,
                      const int (&kind)[3], hipStream_t s);

}  // namespace sps
