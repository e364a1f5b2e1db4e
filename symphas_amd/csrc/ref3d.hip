// ref3d.hip - the reference-order streams of 3D single-field steps.
//
// Compiled with -ffp-contract=off (ref_stream.hpp).  Built for the 7- and
// 15-point laplacians and the 25-point bilaplacian; other stencils, and sets
// without a laplacian, keep the one-site kernel.
#include "term_set.hpp"

namespace sps {
namespace {

template <typename T, int SET, int L>
void launch_set3(const T* in, T* out, const RefParams<T>& p,
                 const int (&kind)[3], hipStream_t s) {
  launch_ref_stream3d<T, 4>(stream_fields(in, out, p),
                            make_term_set<T, SET, L, 25>(p, kind), s);
}

}  // namespace

template <typename T>
bool launch_ref_set3d(int set, const T* in, T* out, const RefParams<T>& p,
                      const int (&kind)[3], hipStream_t s) {
  if ((p.L != 7 && p.L != 15) || ((set & kSBilap) && p.B != 25)) return false;
  if (one_site_step3d(p.n[0], p.n[1], p.n[2], sizeof(T))) return false;
  switch (set) {
#define SPS_SET3(SET)                                        \
  case SET:                                                  \
    if (p.L == 7) launch_set3<T, SET, 7>(in, out, p, kind, s); \
    else launch_set3<T, SET, 15>(in, out, p, kind, s);       \
    return true
    SPS_SET3(kSLap);
    SPS_SET3(kSLapOp);
    SPS_SET3(kSLap | kSLapOp);
    SPS_SET3(kSLap | kSId);
    SPS_SET3(kSLapOp | kSId);
    SPS_SET3(kSLap | kSLapOp | kSId);
    SPS_SET3(kSLap | kSBilap);
    SPS_SET3(kSLapOp | kSBilap);
    SPS_SET3(kSLap | kSLapOp | kSBilap);
    SPS_SET3(kSLap | kSBilap | kSId);
    SPS_SET3(kSLapOp | kSBilap | kSId);
#undef SPS_SET3
    default: return false;
  }
}

template bool launch_ref_set3d<float>(int, const float*, float*,
                                      const RefParams<float>&, const int (&)[3],
                                      hipStream_t);
template bool launch_ref_set3d<double>(int, const double*, double*,
                                       const RefParams<double>&,
                                       const int (&)[3], hipStream_t);

}  // namespace sps
