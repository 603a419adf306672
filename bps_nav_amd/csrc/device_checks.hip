// Parts of the library that tests call by themselves, device functions over whole ranges of arguments, which no scene
// reaches, and rules of the host's: a library of its own (libbpsx_checks.so) that nothing but the tests loads.
#include <hip/hip_runtime.h>

#include "geodesic_device.h"
#include "stage_rule.h"
#include "wait_rule.h"

namespace {
// the two roots of bits first + i and first + n - 1 - i, a lane per i
__global__ __launch_bounds__(256) void k_roots(uint32_t first, uint32_t n, float* a, float* b) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  bpsx::sqrt_exact2(__uint_as_float(first + i), __uint_as_float(first + n - 1u - i), &a[i], &b[n - 1u - i]);
}
// the records of `slot`'s log, `n` of them, applied to the heap that it keeps, of size[0] entries and size[1] - 1 nodes so far
__global__ __launch_bounds__(64) void k_replay(bpsx::GeoSlot* slot, int n, int* size) {
  using namespace bpsx::geo;
  __shared__ GeoShared lds;
  GeoWave g;
  g.lane = (int)threadIdx.x;
  g.L = &lds.a;
  g.ws = slot;
  g.nodeCount = 0;
  bpsx::AstarState st;
  st.synced = 0;
  st.logEnd = n;
  st.replaySize = size[0];
  st.replayNodes = size[1];
  replay_log(g, st);
  if (threadIdx.x == 0) { size[0] = st.replaySize; size[1] = st.replayNodes; }
}
}  // namespace

// The reference's heap of `size` entries (total's bits, packed node; entry 1 the root, entry 0 unused, room for 384) after a log of
// n records, `nodes` nodes having been created before it.  Host pointers; returns the entries, or -1 for what no search keeps.
extern "C" __attribute__((visibility("default"))) int bpsx_check_replay(uint32_t* entries, int size, int nodes, const uint32_t* log, int n) {
  constexpr size_t kEntries = 384 * sizeof(uint2);
  if (size < 1 || size > bpsx::geo::kHeapLds || nodes < 1 || nodes > bpsx::kMaxNodes || n < 1 || n > bpsx::kOpLogCap) return -1;
  bpsx::GeoSlot* slot = nullptr;
  int* dsize = nullptr;
  int sizes[2] = {size, nodes};
  const bool ok = hipMalloc(&slot, sizeof(*slot)) == hipSuccess && hipMalloc(&dsize, sizeof(sizes)) == hipSuccess &&
                  hipMemcpy(slot->heap_spill, entries, kEntries, hipMemcpyHostToDevice) == hipSuccess &&
                  hipMemcpy(slot->oplog, log, (size_t)n * sizeof(bpsx::OpRec), hipMemcpyHostToDevice) == hipSuccess &&
                  hipMemcpy(dsize, sizes, sizeof(sizes), hipMemcpyHostToDevice) == hipSuccess;
  if (ok) hipLaunchKernelGGL(k_replay, dim3(1), dim3(64), 0, nullptr, slot, n, dsize);
  const bool done = ok && hipGetLastError() == hipSuccess && hipMemcpy(sizes, dsize, sizeof(sizes), hipMemcpyDeviceToHost) == hipSuccess &&
                    hipMemcpy(entries, slot->heap_spill, kEntries, hipMemcpyDeviceToHost) == hipSuccess;
  (void)hipFree(slot);
  (void)hipFree(dsize);
  return done ? sizes[0] : -1;
}

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

// A wait for a word that comes at look `comes` (0: never), and with `drained` when the device has nothing left to do; the stream answers
// the i-th question, from the look `patience` on, with answers[i], the last of them again and again (StreamIs).  Returns what the wait
// comes to (Wait), and in out the looks, the questions, and how often the device was waited for.
extern "C" __attribute__((visibility("default"))) int bpsx_check_wait(uint32_t comes, int drained, uint32_t patience, const int* answers, uint32_t n, uint32_t* out) {
  struct {
    uint32_t comes, patience, n, looks, asked, drains;
    int drained;
    const int* answers;
    bool heard() { ++looks; return (comes && looks >= comes) || (drains && drained > 0); }
    bool patient() const { return looks < patience; }
    bpsx::StreamIs stream() { return (bpsx::StreamIs)answers[asked++ < n ? asked - 1u : n - 1u]; }
    bool drain() { ++drains; return drained >= 0; }
    void pause() const {}
    void yield() const {}
  } rt{comes, patience, n, 0, 0, 0, drained, answers};
  const int r = (int)bpsx::wait_for_word(rt);
  out[0] = rt.looks; out[1] = rt.asked; out[2] = rt.drains;
  return r;
}
