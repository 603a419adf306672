// How the host waits for a launch that tells of its end by a word in pinned memory (engine.hip, wait_to_be_told).
//
// It looks at the word, and after two milliseconds at the stream as well, which says if a launch has failed.  The stream may have been
// given work behind the launch: that is not waited for.  It may be gone, too: then only the device can say.  Once either has
// nothing left to do the word is there, or the launch has not run: then what it was to write is not there.
#pragma once

namespace bpsx {

enum class StreamIs { kBusy, kIdle, kGone, kFailed };
enum class Wait { kTold, kNeverTold, kFailed };

// rt: heard() of the word, patient() while the stream is not asked yet, stream() -> StreamIs, drain() of the device -> false if that
// failed, pause() between looks, yield() between questions
template <class Runtime> Wait wait_for_word(Runtime& rt) {
  for (unsigned n = 1; !rt.heard(); ++n) {
    rt.pause();
    if (n % 256u || rt.patient()) continue;
    const StreamIs is = rt.stream();
    if (is == StreamIs::kBusy) { rt.yield(); continue; }
    if (is == StreamIs::kFailed) return Wait::kFailed;
    if (rt.heard()) break;
    if (!rt.drain()) return Wait::kFailed;
    return rt.heard() ? Wait::kTold : Wait::kNeverTold;
  }
  return Wait::kTold;
}

}  // namespace bpsx
