// device_math.hip — the kernels' own arithmetic helpers, one value per thread, for the tests
// that compare them with the host's IEEE operations.
#include "kf_device.hpp"
#include "kf_pose_math.hpp"
#include "kf_prior_net.hpp"

namespace {

constexpr int kThreads = 256;

// Float patterns first, first + step, ... (n of them, a multiple of kThreads).
__global__ __launch_bounds__(kThreads) void reciprocals(uint32_t first, uint32_t step, float* out) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  out[i] = kf::reciprocal(__uint_as_float(first + step * i));
}

__global__ __launch_bounds__(kThreads) void bf16s(uint32_t first, uint32_t step, uint16_t* out) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  out[i] = kf::bf16_rne(__uint_as_float(first + step * i));
}

__global__ __launch_bounds__(kThreads) void pivots(const double* in, double* out) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  out[i] = kf::pivot_inverse(in[i]);
}

bool whole_blocks(uint32_t n) { return n != 0 && n % kThreads == 0; }

}  // namespace

extern "C" int dm_reciprocals(uint32_t first, uint32_t step, uint32_t n, float* d_out) {
  if (!whole_blocks(n)) return -1;
  hipLaunchKernelGGL(reciprocals, dim3(n / kThreads), dim3(kThreads), 0, nullptr, first, step, d_out);
  return (int)hipGetLastError();
}

extern "C" int dm_bf16s(uint32_t first, uint32_t step, uint32_t n, uint16_t* d_out) {
  if (!whole_blocks(n)) return -1;
  hipLaunchKernelGGL(bf16s, dim3(n / kThreads), dim3(kThreads), 0, nullptr, first, step, d_out);
  return (int)hipGetLastError();
}

extern "C" int dm_pivots(const double* d_in, uint32_t n, double* d_out) {
  if (!whole_blocks(n)) return -1;
  hipLaunchKernelGGL(pivots, dim3(n / kThreads), dim3(kThreads), 0, nullptr, d_in, d_out);
  return (int)hipGetLastError();
}
