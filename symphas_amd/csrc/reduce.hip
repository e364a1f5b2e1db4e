// reduce.hip - FP64 mass and free-energy sums of a periodic field.
//
// Pass 1: at most kReduceBlocks workgroups, each with a contiguous range of
// rows (y, z); every site contributes psi (mass) and the Landau density of
// energy.hpp (energy), accumulated in FP64 even for FP32 fields
// (reduce_rows.hpp).  Waves reduce with xor shuffles, the waves of a block
// through LDS.  Pass 2: one workgroup adds the partials in a fixed order and
// applies the functional's scale (h^D, or 1/sites for the mean).  The result
// is deterministic for a given field and size, wherever the field lies.
#include <mutex>

#include "fused.hpp"
#include "reduce_rows.hpp"

namespace sps {
namespace {

constexpr int kPass1Threads = 512;

template <typename T, int VEC, bool ALIGNED>
__global__ __launch_bounds__(kPass1Threads) void reduce_pass1(
    const T* __restrict__ f, int dim, int X, int Y, int Z, EnergyParams ep,
    double* partials) {
  // neighbouring ranges share rows: keep them on one XCD
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t rows = (int64_t)Y * Z;
  const int r0 = (int)(rows * b / gridDim.x);
  const int r1 = (int)(rows * (b + 1) / gridDim.x);
  double m = 0.0, e = 0.0;
  reduce_rows<T, VEC, ALIGNED>(f, dim, X, Y, Z, r0, r1, ep, m, e);
  block_sum2<kPass1Threads / 64>(m, e);
  if (threadIdx.x == 0) {
    partials[2 * b] = m;
    partials[2 * b + 1] = e;
  }
}

__global__ __launch_bounds__(256) void reduce_pass2(const double* partials,
                                                    int nb, double escale,
                                                    double* sums) {
  double m = 0.0, e = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) {
    m += partials[2 * i];
    e += partials[2 * i + 1];
  }
  block_sum2<4>(m, e);
  if (threadIdx.x == 0) {
    sums[0] = m;
    sums[1] = e * escale;
  }
}

}  // namespace

template <typename T>
int launch_reduce(const T* f, int dim, const int* n, double h,
                  const EnergyParams& ep, double* partials, double* sums,
                  hipStream_t s) {
  const int X = n[0], Y = n[1], Z = dim == 3 ? n[2] : 1;
  const int rows = Y * Z;
  const int nb = rows < kReduceBlocks ? rows : kReduceBlocks;
  // groups of 16 bytes where they divide the rows, in one load each where the
  // field's address allows it (a caller's may lie anywhere)
  constexpr int kVec = 16 / sizeof(T);
  if (X % kVec != 0)
    reduce_pass1<T, 1, true><<<nb, kPass1Threads, 0, s>>>(f, dim, X, Y, Z, ep, partials);
  else if ((uintptr_t)f % 16 == 0)
    reduce_pass1<T, kVec, true><<<nb, kPass1Threads, 0, s>>>(f, dim, X, Y, Z, ep, partials);
  else
    reduce_pass1<T, kVec, false><<<nb, kPass1Threads, 0, s>>>(f, dim, X, Y, Z, ep, partials);
  const double sites = (double)X * Y * Z;
  reduce_pass2<<<1, 256, 0, s>>>(partials, nb, energy_scale(ep, dim, h, sites),
                                 sums);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("reduction launch failed: %s", hipGetErrorString(e));
    return SPS_E_HIP;
  }
  return SPS_OK;
}

template int launch_reduce<float>(const float*, int, const int*, double,
                                  const EnergyParams&, double*, double*,
                                  hipStream_t);
template int launch_reduce<double>(const double*, int, const int*, double,
                                   const EnergyParams&, double*, double*,
                                   hipStream_t);

}  // namespace sps

// ---------------------------------------------------- allocation-free sums
// sps_fd_reduce_device runs the two passes above with their partials in a
// file-scope device array instead of plan memory, so it calls no allocator.
// Pass 1 never uses more than kReduceBlocks workgroups, so this fixed 16 KiB
// holds the partials of a field of any size.  Each GPU holds its own copy of
// the array; host code reaches it only through the address that
// hipGetSymbolAddress returns for the current device (the array's name is a
// host-side stand-in, not a device address).
namespace sps {
namespace {

__device__ __align__(256) double scratch[2 * kReduceBlocks];

constexpr int kScratchDevices = 64;
std::mutex scratch_mu;
double* scratch_dev[kScratchDevices] = {};

// Address of the current device's scratch array, looked up once per device.
int scratch_address(double** out) {
  int dev = -1;
  SPS_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kScratchDevices) {
    set_error("device %d beyond the %d devices the scratch table covers", dev,
              kScratchDevices);
    return SPS_E_HIP;
  }
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_dev[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_error("hipGetSymbolAddress(scratch) on device %d failed: %s", dev,
                hipGetErrorString(e));
      return SPS_E_HIP;
    }
    scratch_dev[dev] = static_cast<double*>(ptr);
  }
  *out = scratch_dev[dev];
  return SPS_OK;
}

}  // namespace
}  // namespace sps

extern "C" int sps_fd_reduce_device(int dim, int dtype, const int32_t* n,
                                    double h, const sps_fd_energy* energy,
                                    const void* field, double* sums,
                                    void* hip_stream) {
  using namespace sps;
  // every argument is checked before the first HIP call
  if (dim != 2 && dim != 3) {
    set_error("dim must be 2 or 3 (got %d)", dim);
    return SPS_E_INVALID;
  }
  if (dtype != SPS_F32 && dtype != SPS_F64) {
    set_error("dtype must be SPS_F32 or SPS_F64 (got %d)", dtype);
    return SPS_E_INVALID;
  }
  if (!n || !field || !sums) {
    set_error("n, field and sums must not be NULL");
    return SPS_E_INVALID;
  }
  double sites = 1.0;
  for (int a = 0; a < dim; ++a) {
    if (n[a] < 1 || n[a] > (1 << 20)) {
      set_error("n[%d] = %d out of range [1, 2^20]", a, n[a]);
      return SPS_E_INVALID;
    }
    sites *= n[a];
  }
  if (sites > (double)SPS_REDUCE_DEVICE_MAX_SITES) {
    set_error("field of %.0f sites exceeds the maximum of %d sites", sites,
              SPS_REDUCE_DEVICE_MAX_SITES);
    return SPS_E_INVALID;
  }
  if (!(h > 0) || !std::isfinite(h)) {
    set_error("h must be positive and finite");
    return SPS_E_INVALID;
  }
  EnergyParams ep;
  SPS_TRY(make_energy_params(energy, h, ep));
  double* partials = nullptr;
  SPS_TRY(scratch_address(&partials));
  const int nn[3] = {n[0], n[1], dim == 3 ? n[2] : 1};
  hipStream_t s = static_cast<hipStream_t>(hip_stream);
  return dtype == SPS_F32
             ? launch_reduce<float>(static_cast<const float*>(field), dim, nn,
                                    h, ep, partials, sums, s)
             : launch_reduce<double>(static_cast<const double*>(field), dim,
                                     nn, h, ep, partials, sums, s);
}
