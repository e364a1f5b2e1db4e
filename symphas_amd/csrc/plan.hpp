// plan.hpp - the single-field plan behind sps_fd_plan*.
#pragma once

#include "common.hpp"
#include "energy.hpp"
#include "fused.hpp"
#include "shape.hpp"

namespace sps {
void set_error(const char* fmt, ...);
const char* last_error();
int validate_desc(const sps_fd_desc* d);
Lowered lower(const sps_fd_desc& d);
template <typename T>
void make_fused_coef(const sps_fd_desc& d, const Lowered& lw, FusedCoef<T>& c);
// Reference-order parameters of term group `group` (0: the right-hand side,
// k >= 1: the definition of var(k)).
template <typename T>
void make_ref_params(const sps_fd_desc& d, RefParams<T>& p, int group = 0);
void interior_to_padded(const sps_fd_desc& d, const char* src, char* dst,
                        size_t es, bool fill_ghosts);
void padded_to_interior(const sps_fd_desc& d, const char* src, char* dst,
                        size_t es);

// Launches replayed per captured graph (even, so buffer parity is kept).
constexpr int kGraphLaunches = 16;

struct GraphSlot {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};
}  // namespace sps

struct sps_fd_plan {
  sps_fd_desc d{};
  hipStream_t stream = nullptr;      // stream work is enqueued on
  hipStream_t own_stream = nullptr;  // the plan's own stream
  size_t nsites = 0, esize = 0;
  void* buf[2] = {nullptr, nullptr};  // ping-pong fields (unpadded)
  int cur = 0;                        // buf[cur] holds the current field
  void* work = nullptr;               // dframe / derivative output
  double* partials = nullptr;
  double* sums = nullptr;
  sps::EnergyParams energy{};  // functional of sps_fd_reduce
  bool has_data = false;
  int path = SPS_PATH_REFERENCE;
  sps::Lowered low;
  sps::RefParams<float> rp32;   // right-hand side
  sps::RefParams<double> rp64;
  void* vars[SPS_MAX_PROV] = {nullptr, nullptr};  // provisional grids
  sps::RefParams<float> prov32[SPS_MAX_PROV];     // their definitions
  sps::RefParams<double> prov64[SPS_MAX_PROV];
  sps::FusedCoef<float> fc32;
  sps::FusedCoef<double> fc64;
  int K = 1;    // fused: steps per launch
  int TY = 32;  // fused 2D: rows per chunk; fused 3D: y rows per wave
  int TZ = 64;  // fused 3D: planes per chunk
  int VEC = 4;  // fused 2D: values per lane (16 or 8 bytes)
  sps::GraphSlot graphs[2];  // indexed by the buffer parity at capture

  int launch_one(int k);
  // reference-order passes that fill the provisional grids from buf[cur]
  int launch_provisionals();
  int steps_per_launch() const;
  int step(int nsteps);
  void drop_graphs();

  // Launch shape before any tuning (shape.hpp).  2D: four steps per launch,
  // the best at every size measured.  3D at radius one: t of the (steps, rows)
  // shapes as fitted over 32^3 .. 256^3 and uneven boxes.
  void choose_default_shape() {
    const int R = fc64.radius, X = d.n[0], Y = d.n[1], Z = d.n[2];
    sps::StreamShape s;
    if (d.dim == 2) {
      s = sps::stream_shape2d(X, Y, 4, R, (int)esize);
    } else if (R == 2) {
      s = sps::radius_two_shape3d(X, Y, Z, (int)esize);
    } else if (d.dtype == SPS_F32) {
      static const sps::Stream3DCand c[4] = {
          {2, 4, 0.258}, {2, 6, 0.333}, {2, 8, 0.433}, {2, 12, 0.603}};
      s = sps::stream_shape3d(X, Y, Z, R, 4, 1, c, 4, 1.4);
    } else {
      // Two steps of 4 rows always: one step of 8 rows was 18.6 us per step on
      // 61x500x200, two of 4 rows 15.9.  Even splits of Z, the tallest of equal
      // cost (fewer planes read twice where HBM is the bound).
      static const sps::Stream3DCand two = {2, 4, 0.418};
      double least = 0;
      for (int m = 1; m <= Z; ++m) {
        const int tz = (Z + m - 1) / m;
        if (tz > 1024) continue;
        const double cost = sps::stream_cost3d(X, Y, Z, R, 8, 1, two, tz, 1.1);
        if (least == 0 || cost < least * 0.999) {
          least = cost;
          s = sps::StreamShape{2, 4, tz, 1};
        }
      }
    }
    K = s.steps;
    TY = s.rows;
    TZ = d.dim == 3 ? s.planes : 64;
    VEC = d.dim == 2 ? s.vec : 16 / (int)esize;
  }

  int allocate() {
    SPS_HIP_TRY(hipStreamCreateWithFlags(&own_stream, hipStreamNonBlocking));
    stream = own_stream;
    for (int i = 0; i < 2; ++i) {
      hipError_t e = hipMalloc(&buf[i], nsites * esize);
      if (e != hipSuccess) {
        buf[i] = nullptr;
        sps::set_error("hipMalloc of %zu bytes failed: %s", nsites * esize,
                       hipGetErrorString(e));
        return SPS_E_NOMEM;
      }
    }
    SPS_HIP_TRY(hipMalloc(&partials, 2 * sps::kReduceBlocks * sizeof(double)));
    SPS_HIP_TRY(hipMalloc(&sums, 2 * sizeof(double)));
    for (int k = 0; k < d.nprov; ++k) {
      hipError_t e = hipMalloc(&vars[k], nsites * esize);
      if (e != hipSuccess) {
        vars[k] = nullptr;
        sps::set_error("hipMalloc of a provisional grid failed: %s",
                       hipGetErrorString(e));
        return SPS_E_NOMEM;
      }
    }
    // every term list reads var(k) from vars[k - 1]
    for (int k = 1; k <= d.nprov; ++k) {
      rp32.vars[k] = (const float*)vars[k - 1];
      rp64.vars[k] = (const double*)vars[k - 1];
      for (int j = 0; j < d.nprov; ++j) {
        prov32[j].vars[k] = (const float*)vars[k - 1];
        prov64[j].vars[k] = (const double*)vars[k - 1];
      }
    }
    return SPS_OK;
  }
};
