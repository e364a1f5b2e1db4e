// reduce_rows.hpp - the device part of the FP64 mass and energy sums.
#pragma once

#include "energy.hpp"
#include "lanes.hpp"

namespace sps {

// Adds the sites of rows [r0, r1) (row = y + Y*z) of an X x Y x Z field to m
// (psi) and e (Landau density); the block's threads share the work.  A thread
// takes VEC consecutive sites at a time: their values and the rows above come
// as one load each, and the one x neighbour that is not among them as another.
// With a scalar load per value and neighbour the sums of 512^3 FP32 took 0.58
// ms (0.9 TB/s), on latency; this way 0.18 ms.  X must be a multiple of VEC and
// f aligned to VEC values, or ALIGNED false: the same groups, and so the same
// order of the sums, loaded value by value.  Z = 1 in 2D.
template <typename T, int VEC, bool ALIGNED = true>
__device__ __forceinline__ void reduce_rows(const T* __restrict__ f, int dim,
                                            int X, int Y, int Z, int r0, int r1,
                                            const EnergyParams& ep, double& m,
                                            double& e) {
  const int g = X / VEC;
  const int nthreads = blockDim.x;
  // position of this thread's group, advanced by nthreads groups a time
  const int dr = nthreads / g, dx = nthreads - dr * g;
  int xg = threadIdx.x % g;
  int r = r0 + (int)(threadIdx.x / g);
  int y = r % Y, z = r / Y;
  const bool central = ep.central != 0;
  const int64_t XY = (int64_t)X * Y;
  auto load = [](const T* p, T (&v)[VEC]) {
    if constexpr (ALIGNED) {
      load_vec<VEC>(p, v);
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[j] = p[j];
    }
  };
  while (r < r1) {
    const int x = xg * VEC;
    const T* row = f + (int64_t)r * X;
    T v[VEC], up[VEC], dn[VEC];
    load(row + x, v);
    load((y + 1 == Y ? row - (XY - X) : row + X) + x, up);
    const T right = row[x + VEC == X ? 0 : x + VEC];
    T left = v[0];
    double g2[VEC];
    if (central) {
      left = row[x == 0 ? X - 1 : x - 1];
      load((y == 0 ? row + (XY - X) : row - X) + x, dn);
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      // the backward neighbour is the site itself for the forward difference
      const T xp = central ? (j == 0 ? left : v[j - 1]) : v[j];
      const double gx = (double)(j + 1 < VEC ? v[j + 1] : right) - (double)xp;
      const double gy = (double)up[j] - (double)(central ? dn[j] : v[j]);
      g2[j] = gx * gx + gy * gy;
    }
    if (dim == 3) {
      load((z + 1 == Z ? f + (int64_t)y * X : row + XY) + x, up);
      if (central) load((z == 0 ? row + (Z - 1) * XY : row - XY) + x, dn);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const double gz = (double)up[j] - (double)(central ? dn[j] : v[j]);
        g2[j] += gz * gz;
      }
    }
    double ms = 0.0, es = 0.0;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      ms += (double)v[j];
      es += landau_density(ep, (double)v[j], g2[j]);
    }
    m += ms;
    e += es;
    xg += dx;
    int step = dr;
    if (xg >= g) {
      xg -= g;
      ++step;
    }
    r += step;
    y += step;
    while (y >= Y) {
      y -= Y;
      ++z;
    }
  }
}

// Sum of the block's m and e over its WAVES waves, in thread 0.
template <int WAVES>
__device__ __forceinline__ void block_sum2(double& m, double& e) {
  __shared__ double sh[2][WAVES];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    m += __shfl_xor(m, o, 64);
    e += __shfl_xor(e, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[0][threadIdx.x >> 6] = m;
    sh[1][threadIdx.x >> 6] = e;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    m = e = 0.0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      m += sh[0][w];
      e += sh[1][w];
    }
  }
}

}  // namespace sps
