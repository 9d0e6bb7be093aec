// How the wavefronts of a restore in one launch (fkv_copy_layers_kernel) count what has landed
// and announce the batches of layers.  Free of anything but atomics on the launch's words, so
// that it can also be exercised on host threads.
#pragma once

#include "fkv_internal.h"

namespace fkv {

// One wavefront's part.  Wavefronts run on from batch to batch and the last ranges of several
// batches are under way together, so a batch may be announced before an earlier one: whoever
// waits for a batch looks at the words of all up to it.  (Announced in order, by a count that
// is passed on from batch to batch, eight batches of 256 KiB that land within 36 us took 81
// instead of 71 us.)
struct Landing {
  const LayersLaunch &t;
  const bool first_lane;
  int copied = -1;     // batch of the range this wavefront has copied but not counted yet (-1: none)
  int counted = -1;    // the one whose count is under way
  uint32_t before = 0; // first lane: ranges of it that had landed before

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

  // Whoever has counted the last range of a batch.  The other wavefronts' counts lie behind a
  // release of what they wrote; the acquire makes what they wrote part of what the words release.  (On this
  // chip each of them has written its L2 back before it counted, and nothing would be missing.)
  __device__ __forceinline__ void announce() {
    if (first_lane && counted >= 0 && before + 1 == (uint32_t)t.ranges) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      __hip_atomic_store(t.arrived + counted, 0u, __ATOMIC_RELAXED, // for the next launch
                         __HIP_MEMORY_SCOPE_AGENT);
      t.tick_host[counted] = (uint64_t)wall_clock64();
      __hip_atomic_store(t.landed + counted, t.epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(t.landed_host + counted, t.epoch, __ATOMIC_RELEASE,
                         __HIP_MEMORY_SCOPE_SYSTEM);
    }
    counted = -1;
  }
};

} // namespace fkv
