// How the host waits for the flags that copies leave in page-locked memory (host_copy.hip).  Host code only.
#pragma once

#include <stdint.h>

namespace mi {

constexpr int kFlagMissing = 1;  // (none of the status codes)

// Until `parts` flags hold `ticket`; 0, kFlagMissing, or what the stream fails with.  (The host spins, as hipMemcpy does: 1024 x 4096 x 4096
// 264 us of a core per call, with hipMemcpy 423.)  Stream has
//   int idle(bool *)  whether nothing of it is known to be under way: copies that run beside one another may be, since the last one
//                     launched need not be the last to end
//   int drain()       waits for everything that it was given.
// Asked now and then, so that a copy that failed ends the wait: only a flag that is missing behind drain() is missing.
template <typename Stream>
int await_flags(const uint32_t *flags, int parts, uint32_t ticket, Stream &&stream) {
  auto there = [&](int w) { return __atomic_load_n(flags + w, __ATOMIC_ACQUIRE) == ticket; };
  for (int w = 0, spins = 0; w < parts;) {
    if (there(w)) {
      ++w;
    } else if ((++spins & 0x3fff) != 0) {
      __builtin_ia32_pause();
    } else {
      bool idle = false;
      if (const int rc = stream.idle(&idle)) return rc;
      if (!idle) continue;
      if (const int rc = stream.drain()) return rc;
      while (w < parts && there(w)) ++w;
      return w == parts ? 0 : kFlagMissing;
    }
  }
  return 0;
}

}  // namespace mi
