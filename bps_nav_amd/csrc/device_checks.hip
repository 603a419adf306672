// Device functions that tests call over whole ranges of arguments, which no scene reaches: a library of its own
// (libbpsx_checks.so) that nothing but the tests loads.
#include <hip/hip_runtime.h>

#include "geodesic_device.h"

namespace {
// the two roots of bits first + i and first + n - 1 - i, a lane per i
__global__ __launch_bounds__(256) void k_roots(uint32_t first, uint32_t n, float* a, float* b) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  bpsx::sqrt_exact2(__uint_as_float(first + i), __uint_as_float(first + n - 1u - i), &a[i], &b[n - 1u - i]);
}
}  // namespace

// a[i] = b[i] = the root of the float with bits first + i, each by another of sqrt_exact2's arguments, i < n.
// Device pointers to n floats; returns hipSuccess or the launch's error.
extern "C" __attribute__((visibility("default"))) int bpsx_check_roots(uint32_t first, uint32_t n, float* a, float* b, void* hip_stream) {
  if (!n) return (int)hipSuccess;
  hipLaunchKernelGGL(k_roots, dim3((n - 1u) / 256u + 1u), dim3(256), 0, (hipStream_t)hip_stream, first, n, a, b);
  return (int)hipGetLastError();
}
