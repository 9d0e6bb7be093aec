// How the wavefronts of a restore in one launch (fkv_copy_layers_kernel) count what has landed
// and announce the batches of layers.  Free of anything but atomics on the launch's words, so
// that it can also be exercised on host threads.
#pragma once

#include "fkv_internal.h"

namespace fkv {

// One wavefront's part.  Wavefronts run on from batch to batch and the last ranges of several
// batches are under way together, but a batch is announced only behind the one before it: whoever
// waits for a batch has all earlier ones too, as with a launch per batch on one stream.  That
// the batch before has been announced counts like a range of its own; nobody waits for it, who
// completes a count announces that batch and passes the word on to the next.
struct Landing {
  const LayersLaunch &t;
  const bool first_lane;
  int copied = -1;     // batch of the range this wavefront has copied but not counted yet (-1: none)
  int counted = -1;    // the one whose count is under way
  uint32_t before = 0; // first lane: what had been counted of it before

  __device__ __forceinline__ Landing(const LayersLaunch &t, bool first_lane)
      : t(t), first_lane(first_lane) {}

  // The stores of the copied range have completed (the caller has waited for them).
  __device__ __forceinline__ void count() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent"); // out of this XCD's L2
    if (first_lane)
      before = __hip_atomic_fetch_add(t.arrived + copied, 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
    counted = copied;
    copied = -1;
  }

  // Whoever has completed a count.
  __device__ __forceinline__ void announce() {
    if (first_lane && counted >= 0) {
      int b = counted;
      uint32_t had = before;
      while (had + 1 == (uint32_t)t.ranges + (b > 0 ? 1u : 0u)) {
        t.arrived[b] = 0; // for the next launch
        t.tick_host[b] = (uint64_t)wall_clock64();
        __hip_atomic_store(t.landed + b, t.epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(t.landed_host + b, t.epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        if (++b == t.batches)
          break;
        had = __hip_atomic_fetch_add(t.arrived + b, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    counted = -1;
  }
};

} // namespace fkv
