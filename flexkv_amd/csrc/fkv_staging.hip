// Variable-size chunks between a dense device staging buffer and the host cache,
// with a size table on the host side, and the table of chunk addresses a batched
// codec works on.  The codec-independent device half of a compressed transfer:
// replaces staging_transfer_kernel<is_write_cpu> and build_gpu_chunk_ptrs_kernel<Type>
// of the reference (csrc/compression/common/staging_transfer.cuh:16-122; callers
// csrc/compression/ans/nvcomp_ans.cu:355-409, 455-500).  The codec itself (nvcomp
// ANS) has no counterpart here.
//
// Chunk i of a batch is chunk g = batch_start + i of the call, numbered layer-major,
// then K/V, then block position:  layer = g / (kv_dim * num_blocks),
// kv = (g % (kv_dim * num_blocks)) / num_blocks, b = g % num_blocks.  Its payload
// sits at staging + i * staging_stride, its host slot at
// cpu + (start_layer + layer) * layer_stride + kv * kv_stride + cpu_ids[b] * block_stride,
// its size at size_table[cpu_ids[b] * table_block_stride +
// (start_layer + layer) * table_layer_stride + kv].
//
// One wavefront per chunk at a time (the reference: one 32-lane warp), 8 vectors of
// 16 bytes in flight per lane, sizes of any byte count (16-byte body + byte tail).
// The copy crosses the host link, so the launch has the shape of the link-bound
// gather/scatter kernel: single-wavefront workgroups, a few dozen of them.
#include "fkv_internal.h"

#include <algorithm>
#include <cstring>

namespace fkv {
namespace {

constexpr int64_t kShortMinBytes = 16 << 20; // calls over fewer bytes of slots are over soon
constexpr int64_t kSliceBytes = 64 * kCopyUnroll * 16;
constexpr int64_t kFewWholeSlices = kSliceBytes * 3 / 2; // most payloads in smaller slots have none

struct StagingKernelArgs {
  uint8_t *staging;
  int64_t staging_stride;
  uint64_t *comp_sizes;       // device, [bsz]
  uint8_t *cpu;               // device-visible alias of the host cache
  int64_t chunk_capacity;
  int32_t *overflow;          // device counter or nullptr
  int64_t cpu_kv_stride, cpu_layer_stride, cpu_block_stride;
  const int64_t *cpu_ids;     // device-visible, [num_blocks]; nullptr: in the launch's arguments
  uint32_t *size_table;       // device-visible alias of the host size table
  int64_t table_block_stride, table_layer_stride; // in entries
  int32_t start_layer, num_blocks, batch_start, bsz;
  uint32_t per_layer;         // chunks of a layer (no fewer than a call has, if they are more)
};

typedef unsigned int vec16 __attribute__((ext_vector_type(4)));

// The end of a payload, less than a slice: N accesses of a lane, 64 vectors apart, of which the last
// reaches up to vector `nvec` (not included), and `tail` bytes behind that vector.  Lanes beyond the end
// move the last vector (byte) once more, the same bytes to the same place, instead of sitting
// out: every load is used, so nothing has to be waited for where this joins the path of whole slices
// (see nothing_in_flight in fkv_kernels.hip).
// (To ThreadSanitizer, under which work-items are threads, that is a race.)
#ifndef __has_feature
#define __has_feature(name) 0
#endif
constexpr bool kAllLanesStore = !__has_feature(thread_sanitizer);
template <int N, bool NTS>
__device__ __forceinline__ void copy_end(const FKV_GLOBAL vec16 *s, FKV_GLOBAL vec16 *d, int nvec, int tail,
                                         int lane) {
  // without a tail the last byte of the last vector
  const int byte = nvec * 16 + (tail ? min(lane, tail - 1) : -1);
  const uint8_t last = *((const FKV_GLOBAL uint8_t *)s + byte);
  vec16 r[N + 1];
  const int end = min(lane + (N - 1) * 64, nvec - 1);
#pragma unroll
  for (int u = 0; u < N; ++u)
    r[u] = __builtin_nontemporal_load(s + (u + 1 < N ? lane + u * 64 : end));
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (!kAllLanesStore && lane + u * 64 >= nvec)
      continue;
    if (NTS)
      __builtin_nontemporal_store(r[u], d + (u + 1 < N ? lane + u * 64 : end));
    else
      d[u + 1 < N ? lane + u * 64 : end] = r[u];
  }
  if (kAllLanesStore || lane < tail)
    *((FKV_GLOBAL uint8_t *)d + byte) = last;
  asm volatile("" ::"i"(N)); // keeps the last stores of the cases apart, which would be merged and wait
}

// The same for a payload without a whole slice but with more than half of one, in the order of adjacent
// vectors.  Slots of 8 KiB, 50-90 % full, hold little else.  Us, and what a 2048^3 GEMM (27) / a streaming kernel (37)
// beside it takes, vectors 64 apart with 32 wavefronts -> this with 24: 24 MiB 373 (69 / 58) -> 355 (52 / 41),
// 48 MiB 697 (72 / 62) -> 672 (55 / 42).
template <bool NTS>
__device__ __forceinline__ void copy_end_runs(const FKV_GLOBAL vec16 *s, FKV_GLOBAL vec16 *d, int nvec, int tail,
                                              int lane) {
  const int byte = nvec * 16 + (tail ? min(lane, tail - 1) : -1);
  const uint8_t last = *((const FKV_GLOBAL uint8_t *)s + byte);
  vec16 r[kCopyUnroll];
#pragma unroll
  for (int u = 0; u < kCopyUnroll; ++u)
    r[u] = s[min(lane * kCopyUnroll + u, nvec - 1)];
#pragma unroll
  for (int u = 0; u < kCopyUnroll; ++u) {
    if (!kAllLanesStore && lane * kCopyUnroll + u >= nvec)
      continue;
    FKV_GLOBAL vec16 *to = d + min(lane * kCopyUnroll + u, nvec - 1);
    if (NTS)
      __builtin_nontemporal_store(r[u], to);
    else
      *to = r[u];
  }
  if (kAllLanesStore || lane < tail)
    *((FKV_GLOBAL uint8_t *)d + byte) = last;
  asm volatile("" ::"i"(16)); // as above
}

// Copies `bytes` from src to dst with one wavefront; VEC16: both are 16-byte aligned.  RUNS: in whole
// slices, and in payloads that come near one, a lane moves adjacent vectors, 128 bytes, so that its stores complete a line of host
// memory (see copy_slice in fkv_kernels.hip); its loads walk through one line, without the
// streaming hint that might let the line go in between.
template <bool VEC16, bool NTS, bool RUNS>
__device__ __forceinline__ void wave_copy(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst,
                                          int64_t bytes, int lane) {
  if (!VEC16) {
    for (int64_t j = lane; j < bytes; j += 64)
      dst[j] = src[j];
    return;
  }
  constexpr int U = kCopyUnroll;
  constexpr int kLane = RUNS ? U : 1, kAccess = RUNS ? 1 : 64;
  const int64_t whole = bytes / (64 * U * 16);
  const int rest = (int)(bytes - whole * 64 * U * 16), nvec = rest / 16, tail = rest & 15;
  const FKV_GLOBAL vec16 *s = (const FKV_GLOBAL vec16 *)src;
  FKV_GLOBAL vec16 *d = (FKV_GLOBAL vec16 *)dst;
  for (int64_t k = 0; k < whole; ++k, s += 64 * U, d += 64 * U) {
    vec16 r[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const FKV_GLOBAL vec16 *from = s + lane * kLane + u * kAccess;
      r[u] = RUNS ? *from : __builtin_nontemporal_load(from);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      FKV_GLOBAL vec16 *to = d + lane * kLane + u * kAccess;
      if (NTS)
        __builtin_nontemporal_store(r[u], to);
      else
        *to = r[u];
    }
  }
  if (rest == 0)
    return;
  if (RUNS && whole == 0 && nvec > 64 * U / 2)
    return copy_end_runs<NTS>(s, d, nvec, tail, lane);
  switch ((nvec + 63) / 64) {
  case 1: return copy_end<1, NTS>(s, d, nvec, tail, lane);
  case 2: return copy_end<2, NTS>(s, d, nvec, tail, lane);
  case 3: return copy_end<3, NTS>(s, d, nvec, tail, lane);
  case 4: return copy_end<4, NTS>(s, d, nvec, tail, lane);
  case 5: return copy_end<5, NTS>(s, d, nvec, tail, lane);
  case 6: return copy_end<6, NTS>(s, d, nvec, tail, lane);
  case 7: return copy_end<7, NTS>(s, d, nvec, tail, lane);
  case 8: return copy_end<8, NTS>(s, d, nvec, tail, lane);
  default: return copy_end<0, NTS>(s, d, nvec, tail, lane); // a few bytes
  }
}

// Which is the same for all lanes of a wavefront, where the compiler cannot see it.
__device__ __forceinline__ uint32_t same_for_wave(uint32_t v) {
#if defined(__HIP__)
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
#else
  return v;
#endif
}

// What a payload costs its wavefront besides its bytes is what it waits for: its place and size,
// the bytes behind its last vector, the acknowledgement of its stores.  Ids and sizes come
// through the scalar cache, a payload ahead, which leaves the counter of loads and stores alone; the
// bytes are asked for with the last vectors; stores of whole slices are not waited for.  With all
// that in line (48 MiB of slots 50-90 % full, us, before -> this, wavefronts alike): written from
// slots of 32 KiB 675 -> 656, 8 KiB 700 -> 692, 2 KiB 983 -> 849; read 650 -> 637, 683 -> 644, 1977 -> 1268.
template <bool WRITE_CPU, bool VEC16, bool RUNS = false>
__global__ __launch_bounds__(kCopyBlockThreads) void fkv_staging_transfer_kernel(StagingKernelArgs a,
                                                                                 ArgPlan plan) {
  const FKV_CONSTANT int64_t *const cpu_ids = (const FKV_CONSTANT int64_t *)(
      a.cpu_ids ? a.cpu_ids : reinterpret_cast<const int64_t *>(plan.w));
  const int lane = threadIdx.x & 63;
  const uint32_t wave = blockIdx.x * (blockDim.x / 64) + same_for_wave(threadIdx.x / 64);
  const uint32_t nwaves = gridDim.x * (blockDim.x / 64), bsz = (uint32_t)a.bsz;
  // Where chunk i lives on the host side: (layer, kv) and the id of its block.
  struct Place {
    uint32_t layer, kv;
    int64_t id;
  };
  auto place = [&](uint32_t i) {
    const uint32_t g = (uint32_t)a.batch_start + i;
    const uint32_t layer = g / a.per_layer, in_layer = g - layer * a.per_layer;
    const uint32_t kv = in_layer / (uint32_t)a.num_blocks;
    return Place{layer, kv, cpu_ids[in_layer - kv * (uint32_t)a.num_blocks]};
  };
  auto slot_of = [&](const Place &p) {
    return a.cpu + ((int64_t)p.layer + a.start_layer) * a.cpu_layer_stride + p.kv * a.cpu_kv_stride +
           p.id * a.cpu_block_stride;
  };
  auto entry_of = [&](const Place &p) {
    return a.size_table + p.id * a.table_block_stride +
           (a.start_layer + (int64_t)p.layer) * a.table_layer_stride + p.kv;
  };
  // out of HBM where it is written, out of host memory, a round trip over the link, where it is read
  // (64 bits without a sign: a compressor's "failed" may be the largest of them)
  auto size_of = [&](uint32_t i, const Place &p) -> uint64_t {
    return WRITE_CPU ? ((const FKV_CONSTANT uint64_t *)a.comp_sizes)[i]
                     : (uint64_t)*(const FKV_CONSTANT uint32_t *)entry_of(p);
  };
  if (wave >= bsz)
    return;
  Place here = place(wave), next = place(min(wave + nwaves, bsz - 1));
  uint64_t sz_next = size_of(wave, here);
  for (uint32_t i = wave; i < bsz; i += nwaves) {
    uint8_t *const cur_slot = slot_of(here);
    uint32_t *const cur_entry = entry_of(here);
    const uint64_t sz = sz_next;
    if (i + nwaves < bsz)
      sz_next = size_of(i + nwaves, next);
    here = next;
    next = place(min(i + 2 * nwaves, bsz - 1)); // both far from 2^32
    uint8_t *payload = a.staging + i * a.staging_stride;
    if (WRITE_CPU) {
      if (sz > (uint64_t)a.chunk_capacity) { // does not fit its host slot: counted, size 0 recorded
        if (lane == 0) {
          if (a.overflow)
            atomicAdd(a.overflow, 1);
          *cur_entry = 0;
        }
        continue;
      }
      if (lane == 0)
        *cur_entry = (uint32_t)sz;
      wave_copy<VEC16, false, RUNS>(payload, cur_slot, (int64_t)sz, lane);
    } else {
      if (sz > (uint64_t)a.staging_stride) { // a stale or corrupt entry must not overrun the staging slot
        if (lane == 0) {
          if (a.overflow)
            atomicAdd(a.overflow, 1);
          a.comp_sizes[i] = 0;
        }
        continue;
      }
      if (lane == 0)
        a.comp_sizes[i] = sz;
      wave_copy<VEC16, true, false>(cur_slot, payload, (int64_t)sz, lane);
    }
  }
}

// `base` == nullptr: the table of `planes` base addresses and the ids behind it lie in `plan`.
__global__ void fkv_chunk_ptrs_kernel(void **__restrict__ out, const uint64_t *__restrict__ base,
                                      const int64_t *__restrict__ ids, int64_t block_stride,
                                      int32_t kv_dim, int32_t num_blocks, int32_t batch_start,
                                      int32_t bsz, int32_t planes, ArgPlan plan) {
  if (!base) {
    base = plan.w;
    ids = reinterpret_cast<const int64_t *>(plan.w + planes);
  }
  const int64_t per_layer = (int64_t)kv_dim * num_blocks;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < bsz;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = (int64_t)batch_start + i;
    const int64_t layer = g / per_layer;
    const int64_t kv = (g % per_layer) / num_blocks;
    const int64_t b = g % num_blocks;
    out[i] = reinterpret_cast<void *>(base[layer * kv_dim + kv] + (uint64_t)(ids[b] * block_stride));
  }
}

} // namespace
} // namespace fkv

extern "C" {

int fkv_staging_transfer(const fkv_staging_transfer_desc *dp, void *stream_v) try {
  using namespace fkv;
  clear_error();
  if (!dp)
    return fail(FKV_ERR_INVALID_ARG, "fkv_staging_transfer: null descriptor");
  const fkv_staging_transfer_desc &d = *dp;
  if (d.bsz < 0 || d.batch_start < 0 || d.num_blocks < 1 || d.kv_dim < 1 || d.start_layer_id < 0 ||
      d.staging_stride <= 0 || d.chunk_capacity <= 0)
    return fail(FKV_ERR_INVALID_ARG,
                "fkv_staging_transfer: bsz=%d batch_start=%d num_blocks=%d kv_dim=%d start_layer=%d "
                "staging_stride=%lld chunk_capacity=%lld",
                d.bsz, d.batch_start, d.num_blocks, d.kv_dim, d.start_layer_id,
                (long long)d.staging_stride, (long long)d.chunk_capacity);
  if (d.bsz == 0)
    return FKV_OK;
  if (!d.staging || !d.comp_sizes || !d.cpu_ptr || !d.cpu_block_ids || !d.size_table)
    return fail(FKV_ERR_INVALID_ARG, "fkv_staging_transfer: null pointer");
  for (int i = 0; i < d.num_blocks; ++i)
    if (d.cpu_block_ids[i] < 0)
      return fail(FKV_ERR_INVALID_ARG, "negative block id at position %d", i);
  DeviceGuard guard(d.device);
  if (!guard.ok())
    return fail(FKV_ERR_RUNTIME, "cannot select HIP device %d", d.device);
  int device = 0;
  FKV_HIP_TRY(hipGetDevice(&device));
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  void *cpu_dev = nullptr, *table_dev = nullptr;
  if (hipHostGetDevicePointer(&cpu_dev, d.cpu_ptr, 0) != hipSuccess || !cpu_dev ||
      hipHostGetDevicePointer(&table_dev, d.size_table, 0) != hipSuccess || !table_dev) {
    (void)hipGetLastError();
    return fail(FKV_ERR_INVALID_ARG,
                "fkv_staging_transfer: the host cache and the size table must be device-visible "
                "(pinned or registered)");
  }
  // The ids travel with the launch where they fit (see tables_from_arguments in fkv_kernels.hip),
  // else in plan memory.
  const size_t ids_bytes = (size_t)d.num_blocks * 8;
  PlanSlotHold hold{nullptr, stream};
  uint8_t *dv = nullptr;
  ArgPlan plan;
  if (d.num_blocks <= kArgPlanWords) {
    std::memcpy(plan.w, d.cpu_block_ids, ids_bytes);
  } else {
    hold.slot = plan_acquire(device, ids_bytes);
    if (!hold.slot)
      return FKV_ERR_RUNTIME;
    std::memcpy(plan_host(hold.slot), d.cpu_block_ids, ids_bytes);
    FKV_TRY(plan_publish(hold.slot, ids_bytes, /*mirror=*/true, stream, &dv));
  }
  StagingKernelArgs a{};
  a.staging = static_cast<uint8_t *>(d.staging);
  a.staging_stride = d.staging_stride;
  a.comp_sizes = d.comp_sizes;
  a.cpu = static_cast<uint8_t *>(cpu_dev);
  a.chunk_capacity = d.chunk_capacity;
  a.overflow = d.overflow;
  a.cpu_kv_stride = d.cpu_kv_stride;
  a.cpu_layer_stride = d.cpu_layer_stride;
  a.cpu_block_stride = d.cpu_block_stride;
  a.cpu_ids = reinterpret_cast<const int64_t *>(dv);
  a.size_table = static_cast<uint32_t *>(table_dev);
  a.table_block_stride = d.size_table_block_stride;
  a.table_layer_stride = d.size_table_layer_stride;
  a.start_layer = d.start_layer_id;
  a.num_blocks = d.num_blocks;
  a.batch_start = d.batch_start;
  a.bsz = d.bsz;
  a.per_layer = (uint32_t)std::min<int64_t>((int64_t)d.kv_dim * d.num_blocks, UINT32_MAX);
  const uint64_t align = (uint64_t)(uintptr_t)a.staging | (uint64_t)a.staging_stride |
                         (uint64_t)(uintptr_t)a.cpu | (uint64_t)a.cpu_kv_stride |
                         (uint64_t)a.cpu_layer_stride | (uint64_t)a.cpu_block_stride;
  const bool vec16 = (align & 15u) == 0;
  const bool write_cpu = d.is_write_cpu != 0;
  const fkv_launch_policy pol = policy_of(device);
  const int cta = d.transfer_num_cta > 0 ? d.transfer_num_cta : default_num_cta(!write_cpu);
  // The wavefronts of a plain copy to the host, half as many again for a call that is over soon;
  // from the host also, because a wavefront has one payload in flight, whose last slice is short.
  // 48 MiB of slots of 32 KiB, us, and what a 2048^3 GEMM (alone 27) / a streaming kernel (37) next to it
  // takes: written with 16 / 24 / 32 wavefronts 683 (59 / 43) / 663 (105 / 51) / 654 (160 / 72), read with
  // 12 / 18 / 24 715 (44 / 40) / 643 (54 / 41) / 629 (67 / 43).  The wavefronts that waited for their stores, 48
  // and 32 of them, took 662 (67 / 58) and 637 (50 / 41), of slots of 8 KiB 688 (43 / 42) and 657 (40 / 39)
  // against 672 (55 / 42) and 632 (51 / 41) now: a caller whose own kernels matter more takes 3 CTAs, not 4.
  // Slots shorter than a slice hold less, and as many more wavefronts have the same bytes
  // under way: 48 MiB of slots of 2 KiB written 931 -> 715, read 1268 -> 677.
  const int64_t slots = (int64_t)d.bsz * d.staging_stride;
  const int64_t shorter = std::max<int64_t>(1, std::min<int64_t>(4, kSliceBytes / d.staging_stride));
  int grid = cta * (write_cpu ? pol.d2h_wg_per_cta : pol.h2d_wg_per_cta) * (int)shorter;
  if (!write_cpu || slots < kShortMinBytes)
    grid = grid * 3 / 2;
  // Adjacent vectors per lane on the same terms as the fixed-size kernel: not next to a
  // transfer from the host, where the plain order moves 2 % more in sum.  And only for calls
  // that fill the link for a while: the loads of a slice take longer in this order, which a
  // shorter call waits for.  Slots of 32 KiB, us, plain / adjacent: 8 MiB 128 / 133, 16 MiB 237 / 238,
  // 48 MiB 667 / 656; of 2 KiB the same either way.  Such calls reach the link's rate with fewer wavefronts
  // where most payloads have no whole slice and come near one: 24 and 32 take, 48 MiB of slots of 8 KiB, 672 (55 / 42) and
  // 658 (125 / 65), of 10 KiB 674 (57 / 43) and 661 (115 / 63); of 12 KiB 32 are kept, 665 (71 / 49), with
  // 24 675 (59 / 44).
  const bool runs = pol.d2h_lane_runs == 2 ||
                    (pol.d2h_lane_runs == 1 && slots >= kShortMinBytes &&
                     !(pol.arbiter != 0 && link_direction_busy(device, /*h2d=*/true, stream)));
  if (write_cpu && vec16 && runs && d.staging_stride >= kSliceBytes && d.staging_stride < kFewWholeSlices)
    grid = grid * 3 / 4;
  const int threads = write_cpu ? pol.d2h_wg_threads : pol.h2d_wg_threads;
  grid = std::max(1, std::min(grid, (d.bsz + threads / 64 - 1) / (threads / 64)));
#define FKV_LAUNCH_STAGING(...)                                                               \
  hipLaunchKernelGGL((fkv_staging_transfer_kernel<__VA_ARGS__>), dim3(grid), dim3(threads), 0,  \
                     stream, a, plan)
  if (write_cpu && vec16 && runs)
    FKV_LAUNCH_STAGING(true, true, true);
  else if (write_cpu && vec16)
    FKV_LAUNCH_STAGING(true, true);
  else if (write_cpu)
    FKV_LAUNCH_STAGING(true, false);
  else if (vec16)
    FKV_LAUNCH_STAGING(false, true);
  else
    FKV_LAUNCH_STAGING(false, false);
#undef FKV_LAUNCH_STAGING
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(FKV_ERR_RUNTIME, "staging transfer launch failed: %s", hipGetErrorString(e));
  stats().kernel_launches.fetch_add(1, std::memory_order_relaxed);
  if (d.sync)
    FKV_HIP_TRY(hipStreamSynchronize(stream));
  return FKV_OK;
} catch (...) {
  return fkv::caught(__func__);
}

int fkv_build_gpu_chunk_ptrs(const fkv_chunk_ptrs_desc *dp, void *stream_v) try {
  using namespace fkv;
  clear_error();
  if (!dp)
    return fail(FKV_ERR_INVALID_ARG, "fkv_build_gpu_chunk_ptrs: null descriptor");
  const fkv_chunk_ptrs_desc &d = *dp;
  if (d.backend != FKV_BACKEND_VLLM && d.backend != FKV_BACKEND_TRTLLM &&
      d.backend != FKV_BACKEND_SGLANG)
    return fail(FKV_ERR_RUNTIME, "Unsupported gpu_block_type: %d", d.backend);
  if (d.bsz < 0 || d.batch_start < 0 || d.num_blocks < 1 || d.kv_dim < 1 || d.start_layer_id < 0)
    return fail(FKV_ERR_INVALID_ARG, "fkv_build_gpu_chunk_ptrs: bsz=%d batch_start=%d num_blocks=%d "
                "kv_dim=%d start_layer=%d", d.bsz, d.batch_start, d.num_blocks, d.kv_dim,
                d.start_layer_id);
  if (d.bsz == 0)
    return FKV_OK;
  if (!d.out_ptrs || !d.gpu_tensor_ptrs || !d.gpu_block_ids)
    return fail(FKV_ERR_INVALID_ARG, "fkv_build_gpu_chunk_ptrs: null pointer");
  const int64_t per_layer = (int64_t)d.kv_dim * d.num_blocks;
  const int64_t first_layer = d.batch_start / per_layer;
  const int64_t last_layer = ((int64_t)d.batch_start + d.bsz - 1) / per_layer;
  const int64_t last_abs = d.start_layer_id + last_layer;
  const int64_t need = d.backend == FKV_BACKEND_TRTLLM ? 1
                       : d.backend == FKV_BACKEND_VLLM
                           ? last_abs + 1
                           : (int64_t)(d.kv_dim - 1) * d.num_layers_total + last_abs + 1;
  if (d.num_gpu_tensor_ptrs < need)
    return fail(FKV_ERR_INVALID_ARG, "fkv_build_gpu_chunk_ptrs: %d tensor pointers, %lld needed",
                d.num_gpu_tensor_ptrs, (long long)need);
  for (int i = 0; i < d.num_blocks; ++i)
    if (d.gpu_block_ids[i] < 0)
      return fail(FKV_ERR_INVALID_ARG, "negative block id at position %d", i);
  DeviceGuard guard(d.device);
  if (!guard.ok())
    return fail(FKV_ERR_RUNTIME, "cannot select HIP device %d", d.device);
  int device = 0;
  FKV_HIP_TRY(hipGetDevice(&device));
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  // base addresses of the (layer, kv) planes the batch touches, engine addressing resolved
  const int nplanes = (int)(last_layer + 1) * d.kv_dim;
  const size_t tab = (size_t)nplanes * 8, ids_bytes = (size_t)d.num_blocks * 8;
  const bool carried = (int64_t)nplanes + d.num_blocks <= kArgPlanWords; // as the ids above
  ArgPlan plan;
  PlanSlotHold hold{nullptr, stream};
  uint64_t *h = plan.w;
  if (!carried) {
    hold.slot = plan_acquire(device, tab + ids_bytes);
    if (!hold.slot)
      return FKV_ERR_RUNTIME;
    h = reinterpret_cast<uint64_t *>(plan_host(hold.slot));
  }
  for (int64_t l = 0; l <= last_layer; ++l)
    for (int kv = 0; kv < d.kv_dim; ++kv)
      h[l * d.kv_dim + kv] =
          l < first_layer ? 0
                          : gpu_chunk_addr(d.backend, d.gpu_tensor_ptrs, d.num_layers_total,
                                           d.gpu_kv_stride, d.gpu_block_stride, d.gpu_layer_stride,
                                           d.start_layer_id + l, kv, 0);
  std::memcpy(h + nplanes, d.gpu_block_ids, ids_bytes);
  uint8_t *dv = nullptr;
  int rc = carried ? FKV_OK : plan_publish(hold.slot, tab + ids_bytes, /*mirror=*/true, stream, &dv);
  if (rc == FKV_OK) {
    const int threads = 256;
    const int grid = std::max(1, std::min((d.bsz + threads - 1) / threads, 1024));
    hipLaunchKernelGGL(fkv_chunk_ptrs_kernel, dim3(grid), dim3(threads), 0, stream, d.out_ptrs,
                       reinterpret_cast<const uint64_t *>(dv),
                       carried ? nullptr : reinterpret_cast<const int64_t *>(dv + tab), d.gpu_block_stride,
                       d.kv_dim, d.num_blocks, d.batch_start, d.bsz, nplanes, plan);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
      rc = fail(FKV_ERR_RUNTIME, "chunk pointer launch failed: %s", hipGetErrorString(e));
  }
  if (rc != FKV_OK)
    return rc;
  stats().kernel_launches.fetch_add(1, std::memory_order_relaxed);
  if (d.sync)
    FKV_HIP_TRY(hipStreamSynchronize(stream));
  return FKV_OK;
} catch (...) {
  return fkv::caught(__func__);
}

} // extern "C"
