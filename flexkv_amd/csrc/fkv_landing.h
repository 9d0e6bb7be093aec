// How the wavefronts of a restore in one launch (fkv_copy_layers_kernel) count what has landed
// and announce the batches of layers.  Free of anything but atomics on the launch's words, so
// that it can also be exercised on host threads.
#pragma once

#include "fkv_internal.h"

#include <algorithm>

namespace fkv {

// How a restore of `batches` batches of `pairs_per_batch` (layer, kv) pairs, the last one of
// `last_pairs`, each of `per_pair` slices, is cut for `working` wavefronts.  Ranges of 16 slices
// (128 KiB), or smaller ones where the whole restore would not make two rounds of the wavefronts;
// the last batch, which may be shorter than the others, into ranges of about the same size.  None
// is empty.  A batch need not go round the wavefronts: they run on into the next one.  (Ranges of
// 64 KiB, and as many a batch as there are wavefronts: 32 layers of 1 MiB take 1.3 % longer, 61 of
// 7 MiB 1.5 %; of 256 KiB: 3.7 % longer and 0.9 % less.)
struct LayersCut {
  int64_t ranges = 0, last_ranges = 0; // of a batch, of the last one (no more than that)
  int64_t claims(int64_t batches) const { return ranges * (batches - 1) + last_ranges; }
};
inline LayersCut cut_layers(int64_t batches, int64_t pairs_per_batch, int64_t last_pairs,
                            int64_t per_pair, int64_t working) {
  const int64_t slices = per_pair * pairs_per_batch, one = 1;
  LayersCut c;
  c.ranges = std::min(slices, std::max({one, (2 * working + batches - 1) / batches, slices / 16}));
  c.last_ranges = (c.ranges * last_pairs + pairs_per_batch - 1) / pairs_per_batch;
  return c;
}

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
    if (first_lane && counted >= 0 && before + 1 == t.ranges_of(counted)) {
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
