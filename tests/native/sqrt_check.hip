// Runs the square root that the sparse evaluators use (f_sqrt, sdf_eval.h) by
// itself, for tests/test_gpu_sqrt.py.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../isosurface_amd/csrc/sdf_eval.h"

namespace {

// Floats whose bits are in [first, first + n): how many of their roots differ
// from the compiler's correctly rounded one.  K neighbours a lane.
template <int K>
__global__ __launch_bounds__(256) void k_compare(uint32_t first, uint64_t n,
                                                 unsigned long long* differing) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * 256 * K;
  unsigned long long count = 0;
  for (uint64_t i = (static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x) * K; i < n; i += stride) {
    float x[K], r[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
      x[k] = __builtin_bit_cast(float, first + static_cast<uint32_t>(i + k < n ? i + k : n - 1));
    iso::f_sqrt(x, r);
#pragma unroll
    for (int k = 0; k < K; ++k)
      count += __builtin_bit_cast(uint32_t, r[k]) !=
               __builtin_bit_cast(uint32_t, __builtin_sqrtf(x[k]));
  }
  if (count) atomicAdd(differing, count);
}

// Roots of n values; a lane's second value is another one of the array.
__global__ __launch_bounds__(256) void k_roots(const float* in, float* out, int n) {
  const int i = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (i >= n) return;
  const float x[2] = {in[i], in[n - 1 - i]};
  float r[2];
  iso::f_sqrt(x, r);
  out[i] = r[0];
}

}  // namespace

extern "C" {

// `differing` and the arrays are in host memory.
int sqrt_differing(uint32_t first, uint64_t n, int points, unsigned long long* differing) {
  if (n == 0 || first + n > (uint64_t{1} << 32) || (points != 1 && points != 4) || !differing)
    return hipErrorInvalidValue;
  unsigned long long* count = nullptr;
  hipError_t e = hipMalloc(&count, sizeof *count);
  if (e != hipSuccess) return e;
  *differing = 0;
  e = hipMemcpy(count, differing, sizeof *count, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    if (points == 1)
      hipLaunchKernelGGL(k_compare<1>, dim3(4096), dim3(256), 0, nullptr, first, n, count);
    else
      hipLaunchKernelGGL(k_compare<4>, dim3(4096), dim3(256), 0, nullptr, first, n, count);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(differing, count, sizeof *count, hipMemcpyDeviceToHost);
  (void)hipFree(count);
  return e;
}

int sqrt_roots(const float* in, float* out, int n) {
  if (n <= 0 || !in || !out) return hipErrorInvalidValue;
  const size_t bytes = static_cast<size_t>(n) * sizeof(float);
  float* d = nullptr;
  hipError_t e = hipMalloc(&d, 2 * bytes);
  if (e != hipSuccess) return e;
  e = hipMemcpy(d, in, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_roots, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, nullptr,
                       d, d + n, n);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out, d + n, bytes, hipMemcpyDeviceToHost);
  (void)hipFree(d);
  return e;
}

}  // extern "C"
