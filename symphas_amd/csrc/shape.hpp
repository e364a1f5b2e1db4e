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

#include <algorithm>
#include <cmath>
#include <cstdint>

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

// 3D at radius two.  A program that waits for each run has the launches of one
// plan alone on the chip; one that steps several plans in turn has two or three
// launches overlapping, and then the work counts, not the length of a launch:
// chunks that fill every SIMD once shorten a lone launch and stream more fill.
// So a shape has two costs in us per step,
//     alone:   the longest SIMD's planes x alone[waves on it - 1],
//     in turn: all waves' planes x shared / SIMDs, the HBM traffic of three
//              plans, a launch's share of the chip and the host's 4.1 us,
// fitted over 28 boxes of 32^3 .. 300^3 and uneven sides (rms 4% and 8%).
struct Stream3DWave {
  int steps, rows;
  double alone[3], shared;
};
struct Stream3DCost {
  double alone, in_turn;
};
inline Stream3DCost radius_two_cost3d(int X, int Y, int Z, int esize,
                                      const Stream3DWave& c, int planes) {
  const double bytes = 1.0 * X * Y * Z * esize, traffic = 2.3 * bytes / 5.3e6;
  const int64_t strip = 64 - 4 * c.steps;
  const int64_t waves = ((X + strip - 1) / strip) * ((Y + c.rows - 1) / c.rows) *
                        ((Z + planes - 1) / planes);
  const int64_t w = (waves + kSimds - 1) / kSimds;
  const double walk = planes + 4 * c.steps;
  const double t = w <= 3 ? c.alone[w - 1] : std::max(c.alone[2], c.shared * (double)w);
  const double alone =
      (1.5 + std::max(walk * t, 2 * bytes > 256e6 ? traffic : 0.0)) / c.steps;
  const double shared = std::max(walk * c.shared * (double)waves / kSimds,
                                 6 * bytes > 256e6 ? traffic : 0.0);
  return {alone, std::max(alone / 2.3, std::max(shared, 4.1) / c.steps)};
}
// Two steps of tall waves in one round of resident ones is the measure: another
// shape is taken where it costs no more alone and at least 3% less in turn, the
// one of least cost (alone counts four times).  The least cost alone had been
// the rule, and it lost up to 16% in turn against the measure.  us of 50 steps,
// alone / in turn, with the measure, least alone, this rule: FP64 161x150x97 606
// / 448, 540 / 449, 562 / 416; 100^3 598 / 249, 381 / 298, 383 / 209; 220x61x133
// 598 / 329, 449 / 378, 513 / 307; FP32 200^3 810 / 486, 723 / 547, 810 / 486;
// 61x500x200 1156 / 556, 809 / 582, 838 / 524.
inline StreamShape radius_two_shape3d(int X, int Y, int Z, int esize) {
  static const Stream3DWave f32[4] = {{2, 4, {0.727, 0.991, 1.301}, 0.40},
                                      {2, 6, {0.877, 1.189, 1.636}, 0.49},
                                      {2, 8, {1.045, 1.435, 2.152}, 0.64},
                                      {2, 12, {1.27, 1.869, 2.936}, 0.85}};
  // two FP64 steps hold so many registers that a SIMD's second wave runs after
  // the first
  static const Stream3DWave f64[3] = {{1, 4, {0.62, 0.90, 1.43}, 0.50},
                                      {1, 8, {0.96, 1.60, 3.00}, 0.93},
                                      {2, 4, {0.93, 1.91, 2.87}, 1.00}};
  const Stream3DWave* cand = esize == 4 ? f32 : f64;
  const int ncand = esize == 4 ? 4 : 3;
  const Stream3DWave& tall = cand[ncand - 1];
  const int64_t resident = esize == 4 ? 2 * kSimds : kSimds;
  const int64_t per_chunk = ((X + 55) / 56) * ((Y + tall.rows - 1) / tall.rows);
  const int64_t rounds = std::max<int64_t>(1, resident / per_chunk);
  StreamShape best{2, tall.rows,
                   (int)std::min<int64_t>(1024, std::max<int64_t>(16, (Z + rounds - 1) / rounds)),
                   1};
  const double bytes = 1.0 * X * Y * Z * esize;
  const double hbm = 6 * bytes > 256e6 ? 2.3 * bytes / 5.3e6 : 0.0;
  // The halo rows of low waves are read again from the last-level cache or HBM
  // once both fields outgrow the L2s by far: FP32 256^3, 6 rows 25.5 us per step,
  // 12 rows 24.0; 300x280x260, 8 rows 29.2, 12 rows 27.6.
  const int skip = esize == 8 ? 0 : 2 * bytes > 160e6 ? 3 : 2 * bytes > 100e6 ? 2 : 0;
  auto score = [](const Stream3DCost& c) {
    return std::pow(c.alone, 0.8) * std::pow(c.in_turn, 0.2);
  };
  const Stream3DCost one = radius_two_cost3d(X, Y, Z, esize, tall, best.planes);
  // Past the cache the work counts less (400^3 FP64, 80 planes: 10% less alone,
  // 2% more in turn), and not at all where HBM bounds the measure, or where it
  // is more than a round itself.
  const double bound =
      std::max((2 * bytes > 256e6 ? 1.10 : 0.97) * one.in_turn, hbm / tall.steps);
  // Of equal costs, as where HBM bounds them, the lowest chunks: 512^3 FP32 at 74
  // / 57 / 37 planes 163.4 / 164.3 / 162.5 us per step.
  double least = score(one);
  for (int i = skip; i < ncand; ++i)
    for (int planes = std::min(Z, 1024); planes >= 1; --planes) {
      const int m = (Z + planes - 1) / planes;
      planes = (Z + m - 1) / m;  // even chunks
      const Stream3DCost c = radius_two_cost3d(X, Y, Z, esize, cand[i], planes);
      if (c.alone > one.alone || (c.in_turn > bound && per_chunk <= resident) ||
          score(c) > least * (1 + 1e-9))
        continue;
      least = score(c);
      best = StreamShape{cand[i].steps, cand[i].rows, planes, 1};
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
