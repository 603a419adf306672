// Parts of the library that tests call by themselves, device functions over whole ranges of arguments, which no scene
// reaches, and rules of the host's: a library of its own (libbpsx_checks.so) that nothing but the tests loads.
#include <hip/hip_runtime.h>

#include "geodesic_device.h"
#include "stage_rule.h"

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

// A simulator's batched calls of bytes[i] each, one after the other: held[i] is the pinned memory that call i finds; every
// `refuse`-th allocation fails (0: none).  Returns the allocations made.
extern "C" __attribute__((visibility("default"))) uint32_t bpsx_check_stage(const uint64_t* bytes, uint32_t n, uint32_t refuse, uint64_t* held) {
  bpsx::StageRule rule;
  uint32_t asked = 0, made = 0;
  for (uint32_t i = 0; i < n; ++i) {
    const size_t want = rule.wanted(bytes[i]);
    if (want != rule.held) {
      if (refuse && ++asked % refuse == 0) rule.refused();
      else { rule.holds(want); made++; }
    }
    held[i] = rule.held;
  }
  return made;
}
