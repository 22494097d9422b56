// The end of an iterative solve as the host sees it.  The kernel that decides
// stores a tag, unique in its stream, and whether the solve has ended in
// pinned memory; the host looks for it while work queued before is still
// running, so the device stays busy and few launches are queued after the end.
// A slot is written again kSlots tags later: the host waits for a tag before it
// queues the kernel that writes the slot next.
#pragma once
#include "dev.h"

namespace fvk {

struct DoneSlot {
  unsigned long long *at = nullptr;  // null: nobody looks
  unsigned long long tag = 0;
};
__device__ __forceinline__ void done_store(const DoneSlot &s, bool done) {
  if (s.at) __hip_atomic_store(s.at, s.tag << 1 | (done ? 1ull : 0ull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct DoneWatch {
  static constexpr int kSlots = 4;
  unsigned long long *h = nullptr, tag = 0;
  hipError_t init() {
    const hipError_t e = hipHostMalloc((void **)&h, kSlots * sizeof *h, hipHostMallocDefault);
    for (int k = 0; e == hipSuccess && k < kSlots; ++k) h[k] = 0;
    return e;
  }
  void free() {
    if (h) (void)hipHostFree(h);
    h = nullptr;
  }
  DoneSlot next() {
    ++tag;
    return DoneSlot{h + tag % kSlots, tag};
  }
  // The answer of tag t, at most kSlots - 1 behind the last; the wait ends
  // when the stream has nothing left to run.
  hipError_t wait(hipStream_t s, unsigned long long t, bool &done) const {
    const unsigned long long *w = h + t % kSlots;
    for (unsigned spin = 1;; ++spin) {
      unsigned long long v = __atomic_load_n(w, __ATOMIC_ACQUIRE);
      if (v >> 1 != t) {
        if (spin % 65536) continue;
        const hipError_t e = hipStreamQuery(s);
        if (e == hipErrorNotReady) continue;
        if (e != hipSuccess) return e;
        v = __atomic_load_n(w, __ATOMIC_ACQUIRE);
      }
      done = v >> 1 == t && (v & 1);
      return hipSuccess;
    }
  }
};

}  // namespace fvk
