// How the workgroups of a launch that somebody waits for count what they have copied, and the one
// behind whose report nothing is missing raises the word of the launch.  Free of anything but atomics
// on the launch's counts, so that it can also be exercised on host threads.  One work-item of a
// workgroup calls these.
#pragma once

#include "fkv_internal.h"

namespace fkv {

// Launches to the host: before the first share of a workgroup.
__device__ __forceinline__ void begin_on_xcd(const CopyDone &done, uint32_t xcd) {
  (void)__hip_atomic_fetch_add(&done.count->of_xcd[xcd], (uint64_t)1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

// Launches to the host: behind the last share of a workgroup, the stores of all its shares
// acknowledged by the L2 of its XCD.  How far the XCD has come, for newly_released() once the workgroup has
// released that to the system; 0: another workgroup that is at work on the XCD will.
__device__ __forceinline__ uint64_t leave_xcd(const CopyDone &done, uint32_t xcd, uint32_t mine) {
#if defined(__HIP__)
  constexpr int kOrder = __ATOMIC_RELAXED; // through the one L2
#else // host threads have none
  constexpr int kOrder = __ATOMIC_ACQ_REL;
#endif
  const uint64_t change = (uint64_t)mine * kDoneShare - 1;
  const uint64_t left = __hip_atomic_fetch_add(&done.count->of_xcd[xcd], change, kOrder,
                                               __HIP_MEMORY_SCOPE_AGENT) + change;
  return left % kDoneShare ? 0 : left / kDoneShare;
}

// The shares that are this workgroup's to report: `far` less what has been reported before.
//
// While it was in its release others may have started on the XCD, been the last one at work again and
// reported its shares with theirs; the launch may be over by now, the host gone on, the next launch
// under way with these counts.  Nothing is left for it then, because what has been reported only ever
// grows.  (With counts that start at zero for every launch it found zero there, and reported its shares once
// more, to the next launch.  Taking the shares in the step in which it leaves, a compare-and-swap, is sound too,
// but the workgroups of an XCD leave together and get into each other's way: 10 MiB to the host
// 208.7 us, this 206.2.)
__device__ __forceinline__ uint32_t newly_released(const CopyDone &done, uint32_t xcd, uint64_t far) {
  const uint64_t before = __hip_atomic_fetch_max(&done.count->reported[xcd], far, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
  return before < far ? (uint32_t)(far - before) : 0;
}

// `shares` of the launch's `all` have been copied and released, and reported by nobody else.
__device__ __forceinline__ void report_copied(const CopyDone &done, uint32_t shares, uint32_t all) {
  if (shares == 0)
    return;
  DoneCounts &c = *done.count;
  if (__hip_atomic_fetch_add(&c.all, shares, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + shares != all)
    return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  // For the next launch.
  __hip_atomic_store(&c.all, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(done.word, done.epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

} // namespace fkv
