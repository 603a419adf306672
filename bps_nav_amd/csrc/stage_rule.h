// How much pinned memory a simulator keeps for the host arrays of its batched calls (engine.hip, BatchArrays).
//
// Calls whose arrays fit it pass through it; the others copy.  A new page of pinned memory costs the host 1.5 us when it is first
// written or read, 0.4 ms a megabyte, and an allocation 0.1 to 0.4 ms.  So calls of more than kAtOnce that do not fit
// copy, until they have copied kPays times as much as the largest of them: about what the memory then costs is what copying has
// cost so far.  (With it at once, the first 50000 samples, moves and snaps of a simulator took 2.7 ms instead of 0.7.)
#pragma once
#include <algorithm>
#include <cstddef>

namespace bpsx {

struct StageRule {
  static constexpr size_t kMost = 16u << 20, kAtOnce = 256u << 10, kPays = 8;
  size_t held = 0;      // bytes of pinned memory
  size_t copied = 0;    // bytes that calls which could have fitted have copied since the last growth for such a call
  size_t largest = 0;   // the largest of them

  // Bytes to hold for a call of `bytes`, what is held where nothing changes; the call copies where that is not enough.
  // Half as much again as the largest needs: calls that grow slowly do not allocate each time.
  size_t wanted(size_t bytes) {
    if (bytes <= held || bytes > kMost) return held;
    if (bytes <= kAtOnce) return kAtOnce;
    largest = std::max(largest, bytes);
    if (copied >= kPays * largest) return std::min(kMost, largest + largest / 2);
    copied += bytes;
    return held;
  }
  // what wanted() asked for is there
  void holds(size_t bytes) {
    held = bytes;
    if (bytes > kAtOnce) copied = largest = 0;
  }
  // or was not to be had: the same again before the next attempt
  void refused() { copied = 0; }
};

}  // namespace bpsx
