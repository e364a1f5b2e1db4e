// multi_ref.hip - reference-order kernel of the coupled-field step.
//
// Compiled with -ffp-contract=off like the single-field reference kernels:
// every product and sum rounds as written, so the FP64 instantiation gives
// the oracle's bits.  One thread per interior site computes every field's
// right-hand side from the current fields (terms in descriptor order, the
// reference's stencil groupings, a monomial operand evaluated at each stencil
// point as its temporary grid would hold it) and writes psi_f + dt * rhs_f.
// Periodic neighbours are found by wrapping coordinates.
#include <cstring>

#include "multi.hpp"
#include "ref_stream.hpp"
#include "stencil_ref.hpp"

namespace sps {
namespace {

struct Offsets {
  int64_t xo[5], yo[5], zo[5];  // element offsets of coordinate c-2 .. c+2
};

// The monomial of the term at element offset off: the left-fold product of
// its factors in field order (psi*rho*rho = (psi*rho)*rho), 1 if empty.
template <typename T>
struct MonoSrc {
  const MRefParams<T>* p;
  const MDevTerm<T>* t;
  __device__ __forceinline__ T operator()(int64_t off) const {
    if (t->single >= 0) return p->in[t->single][off];
    T acc = T(1);
    bool started = false;
    for (int f = 0; f < p->nfields; ++f)
      for (int k = 0; k < t->pow[f]; ++k) {
        const T x = p->in[f][off];
        acc = started ? acc * x : x;
        started = true;
      }
    return acc;
  }
};

// (i, j, k) along get_stride<AX>'s direction vectors to grid offsets
// (datatypes/inc/grid.h:537-578): X: (+x, +y, +z); Y: (+y, -x, +z);
// Z: (-z, +y, -x).
template <typename T, int DIM, int AX, class Src>
struct MAcc {
  const Offsets* o;
  Src src;
  __device__ __forceinline__ T operator()(int i, int j, int k) const {
    int dx, dy, dz;
    if (AX == 0) {
      dx = i; dy = j; dz = k;
    } else if (AX == 1) {
      dx = -j; dy = i; dz = k;
    } else {
      dx = -k; dy = j; dz = -i;
    }
    int64_t off = o->xo[dx + 2] + o->yo[dy + 2];
    if (DIM == 3) off += o->zo[dz + 2];
    return src(off);
  }
};

template <typename T, int DIM, int AX, class Src>
__device__ __forceinline__ T gradlap_m(const MRefParams<T>& p, const Offsets& o,
                                       Src s, int component) {
  MAcc<T, DIM, AX, Src> a{&o, s};
  if (DIM == 2) {
    switch (p.G) {
      case 6: return ref::gradlap2_6<T>(a, p.divh3, component);
      case 8: return ref::gradlap2_8<T>(a, p.divh3);
      case 12: return ref::gradlap2_12<T>(a, p.divh3);
      default: return ref::gradlap2_16<T>(a, p.divh3);
    }
  }
  switch (p.G) {
    case 10: return ref::gradlap3_10<T>(a, p.divh3);
    case 12: return ref::gradlap3_12<T>(a, p.divh3);
    case 28: return ref::gradlap3_28<T>(a, p.divh3);
    case 36: return ref::gradlap3_36<T>(a, p.divh3);
    default: return ref::gradlap3_40<T>(a, p.divh3);
  }
}

template <typename T, int DIM, class Src>
__device__ __forceinline__ T derivative_m(const MRefParams<T>& p,
                                          const Offsets& o, Src s, int dop,
                                          int axis, int component) {
  if (dop == SPS_OP_LAP) {
    MAcc<T, DIM, 0, Src> a{&o, s};
    if (DIM == 2)
      return p.L == 5 ? ref::lap2_5<T>(a, p.divh2) : ref::lap2_9<T>(a, p.divh2);
    switch (p.L) {
      case 7: return ref::lap3_7<T>(a, p.divh2);
      case 15: return ref::lap3_15<T>(a, p.divh2);
      case 19: return ref::lap3_19<T>(a, p.divh2);
      case 21: return ref::lap3_21<T>(a, p.divh2);
      default: return ref::lap3_27<T>(a, p.divh2);
    }
  }
  if (dop == SPS_OP_BILAP) {
    MAcc<T, DIM, 0, Src> a{&o, s};
    if (DIM == 2) {
      switch (p.B) {
        case 13: return ref::bilap2_13<T>(a, p.divh4);
        case 17: return ref::bilap2_17<T>(a, p.divh4);
        default: return ref::bilap2_21<T>(a, p.divh4);
      }
    }
    switch (p.B) {
      case 21: return ref::bilap3_21<T>(a, p.divh4);
      case 25: return ref::bilap3_25<T>(a, p.divh4);
      case 41: return ref::bilap3_41<T>(a, p.divh4);
      case 52: return ref::bilap3_52<T>(a, p.divh4);
      default: return ref::bilap3_57<T>(a, p.divh4);
    }
  }
  if (axis == 0) return gradlap_m<T, DIM, 0>(p, o, s, component);
  if (axis == 1 || DIM == 2) return gradlap_m<T, DIM, 1>(p, o, s, component);
  return gradlap_m<T, DIM, 2>(p, o, s, component);
}

__device__ __forceinline__ int wrap(int c, int n) {
  c %= n;
  return c < 0 ? c + n : c;
}

// c in [-2, n + 2): a neighbour at most two sites away.  For n >= 3 one
// conditional add or subtract gives the same index as wrap without an
// integer division.
__device__ __forceinline__ int wrap_near(int c, int n) {
  if (n < 3) return wrap(c, n);
  return c < 0 ? c + n : (c >= n ? c - n : c);
}

template <typename T, int DIM>
__global__ __launch_bounds__(256) void ref_multi_kernel(MRefParams<T> p) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y * blockDim.y + threadIdx.y;
  const int z = blockIdx.z;
  if (x >= p.n[0] || y >= p.n[1]) return;
  const int64_t nx = p.n[0], nxy = (int64_t)p.n[0] * p.n[1];
  Offsets o;
#pragma unroll
  for (int d = -2; d <= 2; ++d) {
    o.xo[d + 2] = wrap_near(x + d, p.n[0]);
    o.yo[d + 2] = (int64_t)wrap_near(y + d, p.n[1]) * nx;
    o.zo[d + 2] = DIM == 3 ? (int64_t)wrap_near(z + d, p.n[2]) * nxy : 0;
  }
  const int64_t idx = x + nx * y + nxy * z;
  for (int f = 0; f < p.nfields; ++f) {
    T acc = T(0);
    for (int t = 0; t < p.nterms[f]; ++t) {
      const MDevTerm<T>& tm = p.terms[f][t];
      MonoSrc<T> src{&p, &tm};
      T val;
      if (tm.op == SPS_OP_ID) {
        val = tm.coeff * src(idx);
      } else {
        val = tm.coeff * derivative_m<T, DIM>(p, o, src, tm.op, tm.axis,
                                               tm.component);
      }
      acc = t == 0 ? val : acc + val;
    }
    // forward Euler per field (examples/solvers/solverft.h:46-50)
    p.out[f][idx] = p.in[f][idx] + p.dt * acc;
  }
}

// ---------------------------------------------------- the step as a row stream
// (ref_stream.hpp).  Two fields x, y; a right-hand side is a list of
// coeff * D[x^a y^b] known at compile time, as the models of the reference's
// MODEL definitions are (examples/models/modeldefinitions.h:74-80,123-136);
// any other list runs ref_multi_kernel.
struct MTermForm {
  int op, a, b;
};
struct MForm {
  int n[2];
  MTermForm t[2][5];
};
constexpr MForm kModelCForm = {
    {4, 4},
    {{{SPS_OP_BILAP, 1, 0}, {SPS_OP_LAP, 1, 0}, {SPS_OP_LAP, 3, 0}, {SPS_OP_LAP, 0, 2}},
     {{SPS_OP_LAP, 0, 1}, {SPS_OP_ID, 0, 1}, {SPS_OP_ID, 0, 3}, {SPS_OP_ID, 1, 1}}}};
constexpr MForm kGrayScottForm = {
    {4, 3},
    {{{SPS_OP_LAP, 1, 0}, {SPS_OP_ID, 1, 2}, {SPS_OP_ID, 0, 0}, {SPS_OP_ID, 1, 0}},
     {{SPS_OP_LAP, 0, 1}, {SPS_OP_ID, 1, 2}, {SPS_OP_ID, 0, 1}}}};
constexpr MForm kTuringForm = {
    {5, 5},
    {{{SPS_OP_LAP, 1, 0}, {SPS_OP_ID, 1, 0}, {SPS_OP_ID, 0, 1}, {SPS_OP_ID, 1, 2},
      {SPS_OP_ID, 1, 1}},
     {{SPS_OP_LAP, 0, 1}, {SPS_OP_ID, 0, 1}, {SPS_OP_ID, 1, 0}, {SPS_OP_ID, 1, 2},
      {SPS_OP_ID, 1, 1}}}};

constexpr bool form_has(const MForm& f, int op) {
  for (int e = 0; e < 2; ++e)
    for (int t = 0; t < f.n[e]; ++t)
      if (f.t[e][t].op == op) return true;
  return false;
}

// x^a y^b as the left fold of its factors in field order, 1 if none
template <int A, int B, typename T>
__device__ __forceinline__ T mono(const T (&x)[2]) {
  if constexpr (A + B == 0) {
    return T(1);
  } else {
    T acc = A > 0 ? x[0] : x[1];
#pragma unroll
    for (int j = 1; j < A; ++j) acc = acc * x[0];
#pragma unroll
    for (int j = A > 0 ? 0 : 1; j < B; ++j) acc = acc * x[1];
    return acc;
  }
}

template <typename T, const MForm& FORM, int L, int B>
struct FormStep {
  static constexpr int NF = 2;
  // operands under a laplacian that are not a field, in order of appearance
  struct LapOps {
    int n = 0;
    int a[10] = {}, b[10] = {};
    constexpr LapOps() {
      for (int e = 0; e < 2; ++e)
        for (int t = 0; t < FORM.n[e]; ++t)
          if (FORM.t[e][t].op == SPS_OP_LAP && FORM.t[e][t].a + FORM.t[e][t].b != 1 &&
              find(FORM.t[e][t].a, FORM.t[e][t].b) < 0) {
            a[n] = FORM.t[e][t].a;
            b[n++] = FORM.t[e][t].b;
          }
    }
    constexpr int find(int pa, int pb) const {
      for (int d = 0; d < n; ++d)
        if (a[d] == pa && b[d] == pb) return d;
      return -1;
    }
  };
  static constexpr LapOps kOps{};
  static constexpr int NLAP = kOps.n;
  T coeff[2][5];
  T divh2, divh4, dt;

  template <int d>
  __device__ __forceinline__ T lap_operand(const T (&x)[2]) const {
    return mono<kOps.a[d], kOps.b[d]>(x);
  }
  template <class A>
  __device__ __forceinline__ void rhs(const A (&F)[2],
                                      const A (&D)[NLAP > 0 ? NLAP : 1],
                                      const T (&x)[2], T (&r)[2]) const {
    static_for<0, 2>([&](auto ec) {
      constexpr int e = decltype(ec)::value;
      T acc = T(0);
      static_for<0, FORM.n[e]>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        constexpr MTermForm m = FORM.t[e][t];
        T v;
        if constexpr (m.op == SPS_OP_ID) {
          v = mono<m.a, m.b>(x);
        } else if constexpr (m.op == SPS_OP_BILAP) {
          static_assert(m.a + m.b == 1, "the bilaplacian of a field");
          v = rs_bilap<B>(F[m.b], divh4);
        } else if constexpr (m.a + m.b == 1) {
          v = rs_lap<L>(F[m.b], divh2);
        } else {
          v = rs_lap<L>(D[kOps.find(m.a, m.b)], divh2);
        }
        acc = t == 0 ? coeff[e][t] * v : acc + coeff[e][t] * v;
      });
      r[e] = acc;
    });
  }
};

template <typename T>
bool is_form(const MRefParams<T>& p, const MForm& f) {
  if (p.nfields != 2) return false;
  for (int e = 0; e < 2; ++e) {
    if (p.nterms[e] != f.n[e]) return false;
    for (int t = 0; t < f.n[e]; ++t)
      if (p.terms[e][t].op != f.t[e][t].op || p.terms[e][t].pow[0] != f.t[e][t].a ||
          p.terms[e][t].pow[1] != f.t[e][t].b)
        return false;
  }
  return true;
}

template <typename T, const MForm& FORM, int L, int B>
void launch_form_lb(const MRefParams<T>& p, hipStream_t s) {
  FormStep<T, FORM, L, B> step;
  RsFields<T, 2> g;
  std::memset(&g, 0, sizeof(g));
  for (int e = 0; e < 2; ++e) {
    for (int t = 0; t < 5; ++t)
      step.coeff[e][t] = t < FORM.n[e] ? p.terms[e][t].coeff : T(0);
    g.in[e] = p.in[e];
    g.out[e] = p.out[e];
  }
  step.divh2 = p.divh2;
  step.divh4 = p.divh4;
  step.dt = p.dt;
  g.X = p.n[0];
  g.Y = p.n[1];
  g.Z = p.n[2];
  if constexpr (L == 5 || L == 9)
    launch_ref_stream2d(g, step, s);
  else  // FP64 rings of two fields hold two rows
    launch_ref_stream3d<T, sizeof(T) == 8 ? 2 : 4>(g, step, s);
}

template <typename T, const MForm& FORM, int L>
void launch_form_l(const MRefParams<T>& p, hipStream_t s) {
  if constexpr (!form_has(FORM, SPS_OP_BILAP)) {
    launch_form_lb<T, FORM, L, 13>(p, s);
  } else {
    if (p.B == 13) launch_form_lb<T, FORM, L, 13>(p, s);
    else if (p.B == 17) launch_form_lb<T, FORM, L, 17>(p, s);
    else launch_form_lb<T, FORM, L, 21>(p, s);
  }
}

// 2D: every stencil; 3D: the 7- and 15-point laplacians, the 25-point
// bilaplacian.
template <typename T, const MForm& FORM>
bool launch_form(const MRefParams<T>& p, int dim, hipStream_t s) {
  if (!is_form(p, FORM)) return false;
  if (dim == 3) {
    if ((p.L != 7 && p.L != 15) || (form_has(FORM, SPS_OP_BILAP) && p.B != 25))
      return false;
    if (p.L == 7) launch_form_lb<T, FORM, 7, 25>(p, s);
    else launch_form_lb<T, FORM, 15, 25>(p, s);
    return true;
  }
  if (p.L == 5) launch_form_l<T, FORM, 5>(p, s);
  else launch_form_l<T, FORM, 9>(p, s);
  return true;
}

}  // namespace

template <typename T>
int launch_ref_multi(const MRefParams<T>& p, int dim, hipStream_t stream) {
  if (launch_form<T, kModelCForm>(p, dim, stream) ||
      launch_form<T, kGrayScottForm>(p, dim, stream) ||
      launch_form<T, kTuringForm>(p, dim, stream))
    return SPS_OK;
  dim3 block(64, 4, 1);
  dim3 grid((p.n[0] + 63) / 64, (p.n[1] + 3) / 4, dim == 3 ? p.n[2] : 1);
  if (dim == 2)
    ref_multi_kernel<T, 2><<<grid, block, 0, stream>>>(p);
  else
    ref_multi_kernel<T, 3><<<grid, block, 0, stream>>>(p);
  return SPS_OK;
}

template int launch_ref_multi<float>(const MRefParams<float>&, int, hipStream_t);
template int launch_ref_multi<double>(const MRefParams<double>&, int,
                                      hipStream_t);

}  // namespace sps
