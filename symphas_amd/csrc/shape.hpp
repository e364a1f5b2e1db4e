// shape.hpp - launch shapes of the streams before any tuning.  Host code only.
//
// A launch of a stream is one wave per (strip, chunk).  Every wave walks the
// rows (2D) or planes (3D) of its chunk plus the pipeline's fill, and a SIMD
// with w waves takes, per row or plane,
//     max(q, w) * t
// where t is the issue time of one wave's row and q*t the latency of one row
// in a lone wave (its dependent chain).  The launch lasts as long as its
// fullest SIMD, so
//     cost = (chunk + fill) * max(q, ceil(waves / SIMDs)) * t / steps,
// which is short chunks on small fields, and on large ones the height that
// gives every SIMD the same number of waves.
#pragma once

#include <cstdint>
#include <algorithm>

namespace sps {

constexpr int64_t kSimds = 1024;  // 256 CUs of 4 SIMDs

struct StreamShape {
  int steps, rows, planes, vec;
};

// 2D: `steps` fused steps of radius R.  8-byte lanes; FP64 also has 16-byte
// lanes (2 values), which halve the strips' halo and cost 1.7 rows.  q = 1.5
// (1.2 for the wide lanes, whose two chains overlap).  Over 64^2 .. 4096^2 and
// uneven sides, FP32 and FP64, radius one and two, one field or two, the
// shapes this picks are within 1% (geometric mean; 4% at worst) of the best of
// steps {1..4} x heights 4..128 x both lane widths: Allen-Cahn FP64 64^2 0.85
// us per step (64-row chunks 3.8), Model B FP32 2048^2 3.55 (32 rows 4.4),
// Gray-Scott FP32 2048^2 4.9 (32 rows 9.1).
inline StreamShape stream_shape2d(int X, int Y, int steps, int R, int esize,
                                  double q = 1.5) {
  const int narrow = 8 / esize;
  StreamShape best{steps, 4, 0, narrow};
  double least = 0;
  for (int vec = narrow; vec <= (esize == 8 ? 2 : narrow); ++vec) {
    if (X % vec != 0) continue;
    const int halo = (steps * R + vec - 1) / vec;
    const int64_t strip = (int64_t)(64 - 2 * halo) * vec;
    const int64_t nstrips = (X + strip - 1) / strip;
    const double t = vec == narrow ? 1.0 : 1.7;
    const double lone = vec == narrow ? q : q * 0.8;
    for (int rows = 4; rows <= 512; ++rows) {
      const int64_t waves = nstrips * ((Y + rows - 1) / rows);
      const double w = (double)((waves + kSimds - 1) / kSimds);
      const double cost = (rows + 2 * steps * R) * std::max(lone, w) * t;
      if (least == 0 || cost < least) {
        least = cost;
        best.rows = rows;
        best.vec = vec;
      }
      if (rows >= Y) break;
    }
  }
  return best;
}

// 3D: the candidates are (steps, rows per wave) with t in us per plane.  A
// launch also takes 3.2 us to start, and no less than its HBM traffic (the
// field read 1.3 times and written once, at the copy rate of 5.3 TB/s) once
// the fields no longer stay in the 256 MB cache.
struct Stream3DCand {
  int steps, rows;
  double t;
};
// us per step
inline double stream_cost3d(int X, int Y, int Z, int R, int esize, int fields,
                            const Stream3DCand& c, int planes, double q) {
  const double bytes = 1.0 * X * Y * Z * esize * fields;
  const double hbm = 2 * bytes > 256e6 ? 2.3 * bytes / 5.3e6 : 0.0;
  const int64_t strip = 64 - 2 * R * c.steps;
  const int64_t waves = ((X + strip - 1) / strip) * ((Y + c.rows - 1) / c.rows) *
                        ((Z + planes - 1) / planes);
  const double w = (double)((waves + kSimds - 1) / kSimds);
  const double run = (planes + 2 * R * c.steps) * std::max(q, w) * c.t;
  return (3.2 + std::max(run, hbm)) / c.steps;
}
inline StreamShape stream_shape3d(int X, int Y, int Z, int R, int esize,
                                  int fields, const Stream3DCand* cand,
                                  int ncand, double q) {
  StreamShape best{1, cand[0].rows, 16, 1};
  double least = 0;
  for (int i = 0; i < ncand; ++i) {
    for (int tz = 1; tz <= 1024; ++tz) {
      const double cost = stream_cost3d(X, Y, Z, R, esize, fields, cand[i], tz, q);
      if (least == 0 || cost < least) {
        least = cost;
        best = StreamShape{cand[i].steps, cand[i].rows, tz, 1};
      }
      if (tz >= Z) break;
    }
  }
  return best;
}

// Whether a 3D reference-order step runs one thread per site: while all its
// workgroups of 64 x 4 sites are resident at once (two per CU in FP32, one in
// FP64), the launch is one chain of loads and sums, where the plane stream walks
// at least six planes.  <15,10,25> Model B, us per step, one site / stream: FP32
// 44^3 (484 workgroups) 7.2 / 7.6, 48^3 (576) 11.5 / 7.6; FP64 36^3 (324) 13.8 /
// 8.3, and 7.9 at 32^3 (256).
inline bool one_site_step3d(int X, int Y, int Z, int esize) {
  const int64_t workgroups = (int64_t)((X + 63) / 64) * ((Y + 3) / 4) * Z;
  return workgroups <= (esize == 4 ? 512 : 256);
}

}  // namespace sps
