// Gather/scatter kernel of the GPU<->CPU KV-block transfer path (gfx950).
//
// Replaces transfer_kv_blocks_kernel / transfer_kv_blocks_kernel_8b of the
// reference (csrc/transfer.cu:45-158) and the ATen index_select / index_copy_
// device kernels its copy-engine strategies call (csrc/ce_transfer.cu:1051,
// 1135, 1257-1259, 1389-1391).  One kernel serves all of them: it copies
// num_blocks * lk chunks, where both endpoints of chunk (pos, i) are
//     base[i] + ids[pos] * stride.
// The host resolves the engine-specific addressing (vLLM / TRT-LLM / SGLang)
// into the two `base` tables, so the device code has no per-engine variant.
//
// Work decomposition.  A chunk is cut into slices of 64 lanes x kCopyUnroll
// vector accesses (8 KiB for 16-byte vectors).  Slices are numbered
// position-major, then (layer, kv), then slice-in-chunk: that is ascending
// address order inside a block-first host block.  Each workgroup owns one
// contiguous run of slice numbers, hence a contiguous run of block positions
// whose ids it stages in LDS (premultiplied by the block strides) together
// with the two base tables; its wavefronts take slices round-robin, so the
// requests a workgroup has in flight target neighbouring addresses.  A
// wavefront issues all kCopyUnroll loads of a slice before the first store, which
// is what keeps enough reads outstanding to cover the host-link latency in
// the host->GPU direction.  Chunks that are no whole number of slices (compressed layer
// groups, small pages) are packed: the 16-byte vectors of all chunks form one
// flat sequence that is cut into full slices regardless of chunk boundaries,
// every lane resolving the chunk of each of its vectors from the LDS tables, so
// that a wavefront keeps a full slice of requests in flight however long the
// chunks are.
//
// Launch shape.  The link is saturated by roughly 200 KB of requests in flight.
// Requests to host memory sit in the memory-request queues of the XCD that
// issued them until the link has served them, and every other kernel on that
// XCD shares those queues: a few fat workgroups (16 wavefronts each) stall
// memory-bound neighbours for the whole duration of the copy, while the same
// number of bytes in flight spread as single-wavefront workgroups over all
// XCDs costs them little.  The link-bound launches therefore use one
// wavefront per workgroup; only the HBM-to-HBM staging pass uses big ones.
// For the same reason a GPU->host and a host->GPU copy that run at the same
// time slow each other down when they share XCDs (62 GB/s in sum against
// 87-90 GB/s on disjoint halves of the chip); `xcd_mask` confines a launch to
// a subset of the XCDs.  Workgroups of a launch go to the XCDs round-robin, but
// the XCD of workgroup 0 differs from launch to launch (it depends on what was
// dispatched before), so a workgroup reads the id of the XCD it actually runs on
// and leaves if that XCD is not selected; the ones that stay share the work by
// claiming ranges from a counter in device memory.
//
// Data moves as raw integer vectors (integer types cannot canonicalise NaN
// payloads of fp8/bf16 data).  Loads are nontemporal: KV bytes are not reused
// by this kernel.  Stores into HBM are nontemporal too; stores into pinned host
// memory are plain, which measured about 1 GB/s faster over the link.
#include "fkv_internal.h"
#include "fkv_landing.h"
#include "fkv_done.h"

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <vector>

namespace fkv {
namespace {

constexpr int kWave = 64;
constexpr int kSliceWgThreads = 256; // workgroup of fkv_copy_slices_kernel
constexpr size_t kSliceLdsBytes = 53 * 1024; // three workgroups fit the 160 KiB of a CU
constexpr int64_t kSliceFewWgBytes = 64ll << 20;

template <int VEC> struct VecType;
template <> struct VecType<16> { typedef unsigned int type __attribute__((ext_vector_type(4))); };
template <> struct VecType<8>  { typedef unsigned int type __attribute__((ext_vector_type(2))); };
template <> struct VecType<4>  { typedef unsigned int type; };
template <> struct VecType<2>  { typedef unsigned short type; };
template <> struct VecType<1>  { typedef unsigned char type; };

// Id of the XCD this wavefront runs on (the low four bits of the register).
__device__ __forceinline__ uint32_t xcd_of_this_wave() {
  uint32_t v;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
  return v & 15u;
}

// Loads are nontemporal (the bytes are not used again), except where the eight
// accesses of a lane walk through one 128-byte line: a streaming hint lets the line go
// between two of them (measured: 5.6 % of the lines fetched from HBM a second time).
template <typename V, bool NT> __device__ __forceinline__ V get(const V *p) {
  const FKV_GLOBAL V *g = (const FKV_GLOBAL V *)p;
  if (NT)
    return __builtin_nontemporal_load(g);
  return *g;
}

template <typename V, bool NT> __device__ __forceinline__ void put(V v, V *p) {
  FKV_GLOBAL V *g = (FKV_GLOBAL V *)p;
  if (NT)
    __builtin_nontemporal_store(v, g);
  else
    *g = v;
}

// Ends a stretch with predicated stores, of which the compiler must think that they left a load
// unused.  It would otherwise wait for everything in flight, the stores of whole slices too,
// wherever such a stretch joins the path of those: a wavefront then asked for its next slice only
// when the last store of the current one had been acknowledged, which over the link takes as long
// as a load.
__device__ __forceinline__ void nothing_in_flight() {
#if defined(__HIP__)
  __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0)
#endif
}

// Which vector of the slice access u of a lane moves.  Ordinarily an access of the
// wavefront covers 64 adjacent vectors (1 KiB).  With LANE_RUNS a lane moves UNR
// adjacent vectors instead, 128 bytes with 16-byte vectors: the stores of a wavefront
// then complete whole 128-byte lines lane by lane, which the link towards pinned host
// memory takes about 1 % faster when nothing comes the other way (8 GiB GPU->host:
// 57.0 against 56.4 GB/s; a pinned hipMemcpy: 57.0), and 2 % slower in sum when the
// other direction is busy (64 requests both ways: 91.2 against 93.0 GB/s).  The launch
// chooses (CopyKernelArgs::lane_runs); the form is a template parameter because a
// kernel that carries both runs the ordinary one slower (55.8 against 56.2 GB/s).
template <int VEC, bool NTS, int UNR, bool LANE_RUNS>
__device__ __forceinline__ void copy_slice(const uint8_t *__restrict__ src,
                                              uint8_t *__restrict__ dst,
                                              int64_t bytes_in_slice, int lane) {
  using V = typename VecType<VEC>::type;
  constexpr int64_t kSliceBytes = (int64_t)kWave * UNR * VEC;
  constexpr int kLaneStep = LANE_RUNS ? UNR : 1, kAccessStep = LANE_RUNS ? 1 : kWave;
  const int first = lane * kLaneStep;
  const V *__restrict__ s = reinterpret_cast<const V *>(src);
  V *__restrict__ d = reinterpret_cast<V *>(dst);
  // launches with deep unroll have whole slices only (checked where they are shaped)
  if (UNR != kCopyUnroll || bytes_in_slice == kSliceBytes) {
    V r[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      r[u] = get<V, !LANE_RUNS>(s + first + u * kAccessStep);
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      put<V, NTS>(r[u], d + first + u * kAccessStep);
  } else {
    // the short last slice of a chunk: same shape, lanes beyond the end sit out
    // (they re-read the last vector rather than branch around the load)
    const int nvec = (int)(bytes_in_slice / VEC);
    V r[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      r[u] = get<V, !LANE_RUNS>(s + min(first + u * kAccessStep, nvec - 1));
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      if (first + u * kAccessStep < nvec)
        put<V, NTS>(r[u], d + first + u * kAccessStep);
    nothing_in_flight();
  }
}

// How the workgroups of a launch come by their work.  Launches with claim counters
// hand it out in `num_claims` ranges that the workgroups claim one after the other,
// so that a workgroup which is slowed down (it shares its XCD with a transfer in the
// other direction, or its CU with a compute kernel) takes fewer; the others give
// workgroup i the i-th of gridDim.x shares.
// A launch confined to some XCDs: workgroups elsewhere leave.  A workgroup of one
// direction that runs on the other direction's XCDs next to that direction's
// traffic moves its range at a third of the rate and holds up the whole launch, so
// none may stay there.  Workgroup 0 is the safety net for a launch of which no
// workgroup landed on a selected XCD: it looks at the claim counter after a while
// and takes over only if nobody has claimed anything.
// Ranges that safety-net workgroups have copied on this device since the process
// started: zero unless launches found none of their workgroups on the selected XCDs.
__device__ unsigned long long g_safety_net_ranges;

struct Shares {
  unsigned long long *claim; // high half: the launch that owns the count, low half: ranges handed out
  uint32_t num_claims, xcd_mask, epoch;
  uint32_t next_claim; // lane 0: asked for before the current range is copied
  uint32_t taken;      // lane 0 of the safety net: ranges it has claimed itself
  bool confined, dynamic, first, safety_net;

  long long wait_ticks; // of the 100 MHz clock, before the safety net looks at the counter

  __device__ __forceinline__ Shares(const CopyKernelArgs &a)
      : claim(reinterpret_cast<unsigned long long *>(a.claim)), num_claims(a.num_claims),
        xcd_mask(a.xcd_mask), epoch(a.epoch), next_claim(0), taken(0),
        confined(a.xcd_mask != 0), dynamic(a.num_claims != 0), first(true),
        safety_net(false), wait_ticks((long long)a.safety_net_wait_us * 100) {}

  // The counter of a launch need not be clean: it counts for this launch from the
  // moment its high half holds the launch's number, and whoever finds another
  // number there starts it at zero.  Returns the counter as found or made.
  __device__ __forceinline__ unsigned long long adopt() const {
    unsigned long long cur = __hip_atomic_load(claim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((uint32_t)(cur >> 32) != epoch) {
      const unsigned long long fresh = (unsigned long long)epoch << 32;
      // lost to another workgroup of this launch: then it is this launch's already
      if (atomicCAS(claim, cur, fresh) == cur)
        cur = fresh;
      else
        cur = __hip_atomic_load(claim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return cur;
  }
  __device__ __forceinline__ uint32_t claim_one() const {
    return (uint32_t)atomicAdd(claim, 1ull);
  }

  // False: this workgroup takes no part.
  __device__ __forceinline__ bool enter(uint32_t *s_claim) {
    if (confined && !((xcd_mask >> xcd_of_this_wave()) & 1u)) {
      if (blockIdx.x != 0)
        return false;
      if (threadIdx.x == 0) {
        // It looks every microsecond, so that it does not outlast a short launch.
        const long long t0 = wall_clock64();
        bool at_work = false;
        while (!at_work && wall_clock64() - t0 < wait_ticks) { // bounded: the constant 100 MHz clock
          __builtin_amdgcn_s_sleep(32);
          const unsigned long long cur =
              __hip_atomic_load(claim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          at_work = (uint32_t)(cur >> 32) == epoch && (uint32_t)cur != 0;
        }
        *s_claim = at_work ? 1u : (uint32_t)adopt();
      }
      __syncthreads();
      if (*s_claim != 0) // the selected XCDs are at work
        return false;
      __syncthreads();
      // It works from the wrong XCD, so only for as long as nobody else claims anything:
      // no claim ahead of time, and a look at the counter before every claim.
      safety_net = true;
      return true;
    }
    // lane 0 keeps the next claim in a register: it is asked for before the current
    // range is copied and has long arrived when the range is done
    if (dynamic && threadIdx.x == 0) {
      (void)adopt();
      next_claim = claim_one();
    }
    return true;
  }

  // The next share [part/parts, (part+1)/parts) of this workgroup; false: none left
  // (the whole workgroup leaves together).
  __device__ __forceinline__ bool next(uint32_t *s_claim, uint32_t *part, uint32_t *parts) {
    if (!dynamic) {
      *part = blockIdx.x;
      *parts = gridDim.x;
      const bool mine = first;
      first = false;
      return mine;
    }
    if (threadIdx.x == 0) {
      if (!safety_net)
        *s_claim = next_claim;
      else if ((uint32_t)__hip_atomic_load(claim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
               taken)
        *s_claim = 0xffffffffu; // the selected XCDs have turned up
      else {
        *s_claim = claim_one(), ++taken;
        if (*s_claim < num_claims)
          atomicAdd(&g_safety_net_ranges, 1ull);
      }
    }
    __syncthreads();
    *part = *s_claim;
    *parts = num_claims;
    __syncthreads(); // everyone has read the claim before it is overwritten
    if (*part >= *parts)
      return false;
    if (threadIdx.x == 0 && !safety_net)
      next_claim = claim_one();
    return true;
  }
};

// Waits for every load and store of a wavefront.
__device__ __forceinline__ void drain_wave() {
#if defined(__HIP__)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#else
  __syncthreads(); // every work-item has got as far
#endif
}

// Behind the last share of a workgroup, `mine` of the launch's `all`: whoever has copied the last
// one tells the thread that waits.
//
// A waiting thread learns it 5 us sooner than from an event behind the launch (an event is a
// command of its own, which the stream takes up when the kernel has been retired), and 10 us
// sooner than with the two more events that plan memory and the link's bookkeeping used to need.  Whole
// calls, event -> word (us): 53 KiB from the host 28.2 -> 17.2, 2 MiB 58.4 -> 52.7, 72 MiB
// 1340 -> 1332; 130 KiB to it 32.3 -> 21.3, 10 MiB 216.4 -> 207.2, 512 MiB 9450 -> 9444; three layer
// groups 808 -> 793; six puts and six gets of 64 MiB at the same time the same.
//
// Into HBM every workgroup releases what it wrote to whatever runs on the device next, and counts
// its shares.  To the host that would be a release to the system, which waits for whatever its XCD has
// under way: with one for each of 16 workgroups of an XCD a copy of 10 MiB took 9 us longer, one of
// 512 MiB, whose workgroups end milliseconds apart, 40.  So there the workgroups of an XCD, which
// share an L2, count among themselves, and the last one at work on it releases for all (fkv_done.h).
// The L2 knows no owners: that one's release writes back every line which is dirty there, and
// waits for every line on its way out of it, evicted ones too, as it must for its own stores, of
// which some may have been evicted.  The others' stores have been acknowledged by that L2 before they
// leave, so they are among those lines.
template <bool TO_HOST> __device__ __forceinline__ void count_started(const CopyDone &done) {
  if (TO_HOST && done.word && threadIdx.x == 0)
    begin_on_xcd(done, xcd_of_this_wave());
}
template <bool TO_HOST>
__device__ __forceinline__ void count_copied(const CopyDone &done, uint32_t mine, uint32_t all) {
  if (!done.word || mine == 0) // the same for the whole workgroup
    return;
  if (TO_HOST)
    drain_wave();
  else
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __syncthreads();
  if (threadIdx.x != 0)
    return;
  if (TO_HOST) {
    const uint32_t xcd = xcd_of_this_wave();
    const uint64_t far = leave_xcd(done, xcd, mine);
    if (far == 0)
      return;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    mine = newly_released(done, xcd, far);
  }
  report_copied(done, mine, all);
}

// Copies the work units of `a` that fall into [num0/den, num1/den) of the job.
// `load_tables`: the base tables of `a` are not in LDS yet.
template <int VEC, bool NTS, int UNR, bool LR>
__device__ __forceinline__ void copy_share(const CopyKernelArgs &a, uint64_t num0, uint64_t num1,
                                           uint64_t den, uint64_t *lds, bool load_tables) {
  uint64_t *s_base_src = lds;
  uint64_t *s_base_dst = lds + a.lk;
  int64_t *s_off_src = reinterpret_cast<int64_t *>(lds + 2 * a.lk);
  int64_t *s_off_dst = s_off_src + kCopyIdTile;

  constexpr int64_t kSliceBytes = (int64_t)kWave * UNR * VEC;
  constexpr uint32_t kPiece = kWave * UNR; // vectors a wavefront moves per step
  const uint32_t slices = (uint32_t)a.slices_per_chunk;
  // Work units.  Normal mode: slices of a chunk, `spp` per block position.  Packed
  // mode (chunks of no whole number of slices): the vectors of all chunks form one flat
  // sequence, cut into pieces of kPiece vectors regardless of chunk boundaries.
  const uint32_t vpc = (uint32_t)(a.chunk_bytes / VEC);  // vectors per chunk
  const uint32_t spp = a.packed ? (uint32_t)a.lk * vpc : (uint32_t)a.lk * slices;
  const uint64_t total_units = (uint64_t)a.num_blocks * spp;
  const uint64_t total = a.packed ? (total_units + kPiece - 1) / kPiece : total_units;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int nwaves = blockDim.x / kWave;

  uint64_t s0 = total * num0 / den;
  uint64_t s1 = total * num1 / den;
  if (a.packed) { // from pieces to vectors
    s0 *= kPiece;
    s1 = s1 * kPiece < total_units ? s1 * kPiece : total_units;
  }
  const bool any = s0 < s1;

  const uint32_t pos_lo = (uint32_t)(s0 / spp);
  const uint32_t pos_hi = any ? (uint32_t)((s1 - 1) / spp) : pos_lo;
  // This work-item's ids of the first tile are asked for before the tables: where the plan is
  // read in place, out of pinned host memory, that is one round trip over the link instead
  // of two.
  int64_t id_src = (int64_t)pos_lo + tid, id_dst = id_src;
  if (any && (uint32_t)tid < min((uint32_t)kCopyIdTile, pos_hi - pos_lo + 1)) {
    if (a.ids_src)
      id_src = a.ids_src[pos_lo + tid];
    if (a.ids_dst)
      id_dst = a.ids_dst[pos_lo + tid];
  }
  if (load_tables) {
    __syncthreads(); // nobody still reads the tables of the job before
    for (int i = tid; i < a.lk; i += blockDim.x) {
      s_base_src[i] = a.base_src[i];
      s_base_dst[i] = a.base_dst[i];
    }
  }
  if (!any)
    return;
  for (uint32_t tile = pos_lo; tile <= pos_hi; tile += kCopyIdTile) {
    const uint32_t n = min((uint32_t)kCopyIdTile, pos_hi - tile + 1);
    __syncthreads(); // previous tile fully consumed; base tables visible
    for (uint32_t i = tid; i < n; i += blockDim.x) {
      const int64_t p = (int64_t)tile + i;
      if (tile != pos_lo || i != (uint32_t)tid) {
        id_src = a.ids_src ? a.ids_src[p] : p;
        id_dst = a.ids_dst ? a.ids_dst[p] : p;
      }
      s_off_src[i] = id_src * a.stride_src;
      s_off_dst[i] = id_dst * a.stride_dst;
    }
    __syncthreads();
    const uint64_t tile_s0 = (uint64_t)tile * spp;
    const uint64_t t0 = s0 > tile_s0 ? s0 : tile_s0;
    const uint64_t tile_s1 = tile_s0 + (uint64_t)n * spp;
    const uint64_t t1 = s1 < tile_s1 ? s1 : tile_s1;
    if (a.packed) {
      using V = typename VecType<VEC>::type;
      const uint32_t lim = (uint32_t)(t1 - tile_s0); // < kCopyIdTile * spp, checked on host
      const uint32_t ulk = (uint32_t)a.lk;
      // distance between two accesses of a lane and between the first accesses of two
      // lanes, in vectors (see copy_slice for the two orders)
      constexpr uint32_t kStep = LR ? 1 : kWave, kLaneStep = LR ? UNR : 1;
      const uint32_t q64 = kStep / vpc, r64 = kStep % vpc; // kStep vectors = q64 chunks + r64
      const uint32_t qlk = q64 / ulk, rlk = q64 % ulk;     // q64 chunks = qlk positions + rlk
      for (uint32_t v0 = (uint32_t)(t0 - tile_s0) + wave * kPiece; v0 < lim;
           v0 += nwaves * kPiece) {
        V r[UNR];
        V *d[UNR];
        // A lane's vectors are kStep apart.  The first one is located by division;
        // each further one by adding the precomputed quotients and remainders of
        // kStep, which costs a few compares instead of two divisions.  Lanes beyond
        // the end stay on their last valid vector and re-read it rather than branch
        // around the load: all loads of a piece are issued back to back, only the
        // stores are predicated.
        uint32_t v = v0 + lane * kLaneStep;
        const uint32_t vc = min(v, lim - 1);
        const uint32_t c = vc / vpc; // chunk inside the tile: position * lk + i
        uint32_t w = vc - c * vpc;
        uint32_t p = c / ulk;
        uint32_t i = c - p * ulk;
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
          if (u > 0) {
            v += kStep;
            uint32_t w2 = w + r64, i2 = i + rlk, p2 = p + qlk;
            if (w2 >= vpc) {
              w2 -= vpc;
              i2 += 1;
            }
            if (i2 >= ulk) {
              i2 -= ulk;
              p2 += 1;
            }
            const bool ok = v < lim;
            w = ok ? w2 : w;
            i = ok ? i2 : i;
            p = ok ? p2 : p;
          }
          const V *src = reinterpret_cast<const V *>(s_base_src[i] + (uint64_t)s_off_src[p]) + w;
          d[u] = reinterpret_cast<V *>(s_base_dst[i] + (uint64_t)s_off_dst[p]) + w;
          r[u] = get<V, !LR>(src);
        }
        if (v0 + kPiece <= lim) {
#pragma unroll
          for (int u = 0; u < UNR; ++u)
            put<V, NTS>(r[u], d[u]);
        } else {
#pragma unroll
          for (int u = 0; u < UNR; ++u)
            if (v0 + u * kStep + lane * kLaneStep < lim)
              put<V, NTS>(r[u], d[u]);
          nothing_in_flight();
        }
      }
      continue;
    }
    for (uint64_t s = t0 + wave; s < t1; s += nwaves) {
      const uint32_t rel = (uint32_t)(s - tile_s0); // < kCopyIdTile * spp, checked on host
      const uint32_t p = rel / spp;
      const uint32_t r = rel - p * spp;
      const uint32_t i = r / slices;
      const uint32_t sl = r - i * slices;
      const int64_t off = (int64_t)sl * kSliceBytes;
      const int64_t left = a.chunk_bytes - off;
      const uint8_t *src =
          reinterpret_cast<const uint8_t *>(s_base_src[i] + (uint64_t)s_off_src[p]) + off;
      uint8_t *dst = reinterpret_cast<uint8_t *>(s_base_dst[i] + (uint64_t)s_off_dst[p]) + off;
      copy_slice<VEC, NTS, UNR, LR>(src, dst, left < kSliceBytes ? left : kSliceBytes, lane);
    }
  }
}

// Tables that travel in the arguments of a launch instead of lying in memory of their own.
//
// What bounds a small call is what happens before its first load: a plan in pinned host memory
// costs every workgroup a round trip over the link (5000 cycles, 2.2 us), a plan in device memory
// a kernel that brings it there (3 us and the 5 to 10 us between two commands of a stream).
// Arguments are written to device memory by the host itself as part of the launch (a lane has
// its words after 500 cycles) for 0.1 us of host time.  Calls, before -> this (us): transforms of a
// few blocks 14.9 -> 9.8, one of 512 MiB (64 pairs, 256 blocks) 180.8 -> 177.0, payloads of 48 MiB
// to the host 872 -> 865; transfers and restores at kernel_plan_publish.  In these launches the
// four pointers of the arguments hold the number of the first word, plus one; 0: no such list.
template <typename T> __device__ __forceinline__ const T *in_arguments(const T *word, const ArgPlan &plan) {
  return word ? reinterpret_cast<const T *>(plan.w + (reinterpret_cast<uintptr_t>(word) - 1)) : nullptr;
}
__device__ __forceinline__ void tables_from_arguments(CopyKernelArgs &a, const ArgPlan &plan) {
  a.base_src = in_arguments(a.base_src, plan);
  a.base_dst = in_arguments(a.base_dst, plan);
  a.ids_src = in_arguments(a.ids_src, plan);
  a.ids_dst = in_arguments(a.ids_dst, plan);
}

template <int VEC, bool NTS, int U, bool LR>
__device__ __forceinline__ void copy_chunks(const CopyKernelArgs &a) {
  extern __shared__ uint64_t lds[];
  __shared__ uint32_t s_claim;
  Shares shares(a);
  if (!shares.enter(&s_claim))
    return;
  bool load_tables = true;
  uint32_t part, parts, copied = 0;
  while (shares.next(&s_claim, &part, &parts)) {
    if (copied == 0)
      count_started<!NTS>(a.done);
    copy_share<VEC, NTS, U, LR>(a, part, part + 1, parts, lds, load_tables);
    load_tables = false;
    ++copied;
  }
  count_copied<!NTS>(a.done, copied, shares.dynamic ? a.num_claims : gridDim.x);
}
template <int VEC, bool NTS, int U, bool LR = false>
__global__ __launch_bounds__(kCopyBlockThreads) void fkv_copy_chunks_kernel(
    CopyKernelArgs a) {
  copy_chunks<VEC, NTS, U, LR>(a);
}
template <bool NTS, bool LR>
__global__ __launch_bounds__(kCopyBlockThreads) void fkv_copy_chunks_args_kernel(CopyKernelArgs a,
                                                                                 ArgPlan plan) {
  tables_from_arguments(a, plan);
  copy_chunks<16, NTS, kCopyUnroll, LR>(a);
}

// A value that is the same for a whole wavefront, where the compiler cannot see it.
__device__ __forceinline__ uint32_t wave_uniform(uint32_t v) {
#if defined(__HIP__)
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
#else // the CPU model of the device: every work-item has its own
  return v;
#endif
}

// The first lane's value in all lanes, where a workgroup is a single wavefront.
__device__ __forceinline__ uint32_t from_first_lane(uint32_t v) {
#if defined(__HIP__)
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
#else
  return cpu_device_model::from_first_work_item(v);
#endif
}

// A launch of one wavefront that waits for what another launch writes.
#if defined(__HIP__)
#define FKV_LAUNCH_BESIDE(kernel, stream, ...)                                                      \
  hipLaunchKernelGGL(kernel, dim3(1), dim3(kWave), 0, stream, __VA_ARGS__)
#else // the CPU model of the device runs one launch at a time, except for these
#define FKV_LAUNCH_BESIDE(kernel, stream, ...)                                                      \
  cpu_device_model::launch_beside(stream, kWave, [=] { (kernel)(__VA_ARGS__); })
#endif

// Launches that HBM bounds (both ends in device memory): a wavefront looks its slice up in the
// tables, moves it and is done; nothing is staged, and no workgroup waits for itself.
//
// Three workgroups a CU where there are enough slices to fill the chip (kSliceLdsBytes of LDS
// that nobody uses keep the others out).  More wavefronts in flight make the reads and writes
// of HBM get in each other's way: 512 MiB of 32 KiB chunks into a dense buffer take 196 us with
// eight workgroups a CU, 190 with four in 48 KiB, 181 with three, 181 with two, which is
// 5.9 TB/s with the upload of the plan (the yardstick copy: 5.8).  A launch of 64 MiB gains
// 3 %, one of 32 MiB nothing, and the scatter of a staged restore, 36 MiB next to the engine's
// own kernels, should not ask for LDS that it does not need: the limit starts at 64 MiB.
//
// The form with the tables in LDS and 16 vectors a lane, which this one replaces for chunks of
// 8 KiB and more, took (us, before -> this): 512 MiB out of 32 KiB chunks 195 -> 181, back
// into them 205 -> 197, one tensor for all layers 187 -> 180; 288 MiB of 18 KiB chunks
// 116 -> 105; 16 MiB 20 -> 14.  16 vectors a lane instead of 8 (hbm_unroll): 512 MiB 195.
template <int UNR> __device__ __forceinline__ void copy_slices(const CopyKernelArgs &a) {
  constexpr int64_t kSliceBytes = (int64_t)kWave * UNR * 16;
  const uint32_t slices = (uint32_t)a.slices_per_chunk, spp = (uint32_t)a.lk * slices;
  const uint64_t total = (uint64_t)a.num_blocks * spp;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t waves = blockDim.x / kWave;
  const uint64_t step = (uint64_t)gridDim.x * waves;
  for (uint64_t s = (uint64_t)blockIdx.x * waves + wave_uniform(threadIdx.x / kWave); s < total;
       s += step) {
    const uint32_t p = total <= 0xffffffffull ? (uint32_t)s / spp : (uint32_t)(s / spp);
    const uint32_t r = (uint32_t)(s - (uint64_t)p * spp);
    const uint32_t i = r / slices;
    const int64_t off = (int64_t)(r - i * slices) * kSliceBytes;
    const int64_t left = a.chunk_bytes - off;
    const uint8_t *src = reinterpret_cast<const uint8_t *>(
        a.base_src[i] + (uint64_t)((a.ids_src ? a.ids_src[p] : (int64_t)p) * a.stride_src) + off);
    uint8_t *dst = reinterpret_cast<uint8_t *>(
        a.base_dst[i] + (uint64_t)((a.ids_dst ? a.ids_dst[p] : (int64_t)p) * a.stride_dst) + off);
    copy_slice<16, true, UNR, false>(src, dst, left < kSliceBytes ? left : kSliceBytes, lane);
  }
}
template <int UNR>
__global__ __launch_bounds__(kSliceWgThreads) void fkv_copy_slices_kernel(CopyKernelArgs a) {
  copy_slices<UNR>(a);
}
template <int UNR>
__global__ __launch_bounds__(kSliceWgThreads) void fkv_copy_slices_args_kernel(CopyKernelArgs a,
                                                                               ArgPlan plan) {
  tables_from_arguments(a, plan);
  copy_slices<UNR>(a);
}

// Several jobs in one launch (the members of one original layer of a multi-group
// restore, which differ in chunk size and strides): the jobs lie one behind the
// other on a line, each as long as its weight (its bytes), and a share of the launch
// is a stretch of that line.  Counters, mask and grid are those of job 0.
// The argument behind the first one of the running kernel, by its place in the argument memory:
// where the pointers into it are chosen in a loop over the jobs, the compiler would first copy
// all of it to scratch memory.
template <typename First> __device__ __forceinline__ const ArgPlan &plan_behind(const ArgPlan &plan) {
#if defined(__HIP__)
  static_assert(sizeof(First) % alignof(ArgPlan) == 0, "no gap between the two arguments");
  return *reinterpret_cast<const ArgPlan *>(
      (const char *)__builtin_amdgcn_kernarg_segment_ptr() + sizeof(First));
#else
  return plan;
#endif
}

// `plan`: nothing, or the tables of all jobs (see tables_from_arguments).
template <int VEC, bool NTS, int U, bool LR, typename... Plan>
__device__ __forceinline__ void copy_jobs(const CopyJobs &t, const Plan &...plan) {
  extern __shared__ uint64_t lds[];
  __shared__ uint32_t s_claim;
  Shares shares(t.job[0]);
  if (!shares.enter(&s_claim))
    return;
  uint64_t line = 0;
  for (int j = 0; j < t.njobs; ++j)
    line += t.weight[j];
  uint32_t part, parts, copied = 0;
  while (shares.next(&s_claim, &part, &parts)) {
    if (copied == 0)
      count_started<!NTS>(t.job[0].done);
    const uint64_t b0 = line * part / parts, b1 = line * (part + 1) / parts;
    uint64_t off = 0;
    for (int j = 0; j < t.njobs; ++j) {
      const uint64_t w = t.weight[j];
      const uint64_t lo = b0 > off ? (b0 - off < w ? b0 - off : w) : 0;
      const uint64_t hi = b1 > off ? (b1 - off < w ? b1 - off : w) : 0;
      if (lo < hi) {
        CopyKernelArgs a = t.job[j];
        (tables_from_arguments(a, plan), ...);
        copy_share<VEC, NTS, U, LR>(a, lo, hi, w, lds, true);
      }
      off += w;
    }
    ++copied;
  }
  count_copied<!NTS>(t.job[0].done, copied, shares.dynamic ? t.job[0].num_claims : gridDim.x);
}
template <int VEC, bool NTS, int U, bool LR = false>
__global__ __launch_bounds__(kCopyBlockThreads) void fkv_copy_jobs_kernel(CopyJobs t) {
  copy_jobs<VEC, NTS, U, LR>(t);
}
template <bool NTS, bool LR>
__global__ __launch_bounds__(kCopyBlockThreads) void fkv_copy_jobs_args_kernel(CopyJobs t, ArgPlan plan) {
  copy_jobs<16, NTS, kCopyUnroll, LR>(t, plan_behind<CopyJobs>(plan));
}

// Puts the tables of a job into `plan`, behind the `*at` words that are taken, and the numbers of
// their words into `a`; a list that lies there already (`jobs` before this one, of a call over
// several layer groups that share their blocks) is not put there again.  False: no room, or the
// host cannot read the tables.
bool into_arguments(CopyKernelArgs &a, const CopyKernelArgs *jobs, int njobs, ArgPlan &plan, int *at) {
  if (!a.host_tables || a.vec != 16)
    return false;
  auto put = [&](const void *from, int n) -> uintptr_t {
    if (n > kArgPlanWords - *at)
      return 0;
    std::memcpy(plan.w + *at, from, (size_t)n * 8);
    *at += n;
    return (uintptr_t)(*at - n + 1);
  };
  auto table = [&](const uint64_t **words) {
    *words = reinterpret_cast<const uint64_t *>(put(*words, a.lk));
    return *words != nullptr;
  };
  auto list = [&](const int64_t **ids) {
    if (!*ids)
      return true;
    for (int j = 0; j < njobs; ++j)
      if (jobs[j].num_blocks == a.num_blocks)
        for (const int64_t *there : {jobs[j].ids_src, jobs[j].ids_dst})
          if (there && std::memcmp(plan.w + (reinterpret_cast<uintptr_t>(there) - 1), *ids,
                                   (size_t)a.num_blocks * 8) == 0) {
            *ids = there;
            return true;
          }
    *ids = reinterpret_cast<const int64_t *>(put(*ids, a.num_blocks));
    return *ids != nullptr;
  };
  return table(&a.base_src) && table(&a.base_dst) && list(&a.ids_src) && list(&a.ids_dst);
}

// A launch whose tables travel in its arguments; false: they do not fit.
bool launch_with_plan(CopyKernelArgs a, int grid, int threads, size_t lds_bytes, hipStream_t stream) {
  ArgPlan plan;
  int words = 0;
  if (!into_arguments(a, nullptr, 0, plan, &words))
    return false;
  if (a.report)
    a.report->in_arguments = true;
#define FKV_LAUNCH_WITH_PLAN(...)                                                             \
  hipLaunchKernelGGL((__VA_ARGS__), dim3(grid), dim3(threads), lds_bytes, stream, a, plan)
  if (a.per_slice && a.unroll == kCopyUnrollDeep)
    FKV_LAUNCH_WITH_PLAN(fkv_copy_slices_args_kernel<kCopyUnrollDeep>);
  else if (a.per_slice)
    FKV_LAUNCH_WITH_PLAN(fkv_copy_slices_args_kernel<kCopyUnroll>);
  else if (a.nt_store)
    FKV_LAUNCH_WITH_PLAN(fkv_copy_chunks_args_kernel<true, false>);
  else if (a.lane_runs)
    FKV_LAUNCH_WITH_PLAN(fkv_copy_chunks_args_kernel<false, true>);
  else
    FKV_LAUNCH_WITH_PLAN(fkv_copy_chunks_args_kernel<false, false>);
#undef FKV_LAUNCH_WITH_PLAN
  return true;
}

template <int VEC>
int launch_vec(const CopyKernelArgs &a, int grid, int threads, size_t lds_bytes,
               hipStream_t stream) {
  if (a.done.used)
    *a.done.used = true;
  if (VEC == 16 && launch_with_plan(a, grid, threads, lds_bytes, stream))
    ;
  else if (VEC == 16 && a.per_slice && a.unroll == kCopyUnrollDeep)
    hipLaunchKernelGGL(fkv_copy_slices_kernel<kCopyUnrollDeep>, dim3(grid), dim3(threads),
                       lds_bytes, stream, a);
  else if (VEC == 16 && a.per_slice)
    hipLaunchKernelGGL(fkv_copy_slices_kernel<kCopyUnroll>, dim3(grid), dim3(threads), lds_bytes,
                       stream, a);
  else if (a.nt_store)
    hipLaunchKernelGGL((fkv_copy_chunks_kernel<VEC, true, kCopyUnroll>), dim3(grid), dim3(threads),
                       lds_bytes, stream, a);
  else if (VEC == 16 && a.lane_runs)
    hipLaunchKernelGGL((fkv_copy_chunks_kernel<16, false, kCopyUnroll, true>), dim3(grid),
                       dim3(threads), lds_bytes, stream, a);
  else
    hipLaunchKernelGGL((fkv_copy_chunks_kernel<VEC, false, kCopyUnroll>), dim3(grid),
                       dim3(threads), lds_bytes, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(FKV_ERR_RUNTIME, "copy kernel launch failed: %s", hipGetErrorString(e));
  if (a.report)
    a.report->announced = a.done.word && !a.per_slice;
  return FKV_OK;
}

} // namespace

namespace {
// Copies a plan from its pinned host slot to the device mirror.
__global__ void fkv_plan_upload_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src,
                                       uint32_t vectors) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < vectors;
       i += gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// Keeps one wavefront busy for `ticks` of the constant 100 MHz clock.
__global__ void fkv_wait_kernel(long long ticks, int *sink) {
  const long long t0 = wall_clock64();
  while (wall_clock64() - t0 < ticks) {
  }
  if (ticks < 0) // never: keeps the loop from being dropped
    *sink = 1;
}
} // namespace

namespace {
__global__ void fkv_xcd_probe_kernel(uint32_t *present) {
  if (threadIdx.x == 0)
    atomicOr(present, 1u << xcd_of_this_wave());
}
} // namespace

int probe_xcds(uint32_t *present_mask) {
  uint32_t *d = nullptr;
  *present_mask = 0;
  FKV_HIP_TRY(hipMalloc(reinterpret_cast<void **>(&d), sizeof(uint32_t)));
  hipError_t e = hipMemset(d, 0, sizeof(uint32_t));
  if (e == hipSuccess) {
    // far more workgroups than XCDs: the dispatcher deals them out round-robin
    hipLaunchKernelGGL(fkv_xcd_probe_kernel, dim3(1024), dim3(64), 0, nullptr, d);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpy(present_mask, d, sizeof(uint32_t), hipMemcpyDeviceToHost);
  (void)hipFree(d);
  if (e != hipSuccess)
    return fail(FKV_ERR_RUNTIME, "XCD probe failed: %s", hipGetErrorString(e));
  return FKV_OK;
}

uint64_t safety_net_ranges_of_current_device() {
  unsigned long long v = 0;
  if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_safety_net_ranges), sizeof(v)) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return v;
}

int launch_plan_upload(void *device_dst, const void *pinned_src, size_t bytes,
                       hipStream_t stream) {
  const uint32_t vectors = (uint32_t)((bytes + 15) / 16);
  if (vectors == 0)
    return FKV_OK;
  const int threads = 256;
  const int grid = (int)std::min<uint32_t>((vectors + threads - 1) / threads, 64);
  hipLaunchKernelGGL(fkv_plan_upload_kernel, dim3(grid), dim3(threads), 0, stream,
                     static_cast<uint4 *>(device_dst), static_cast<const uint4 *>(pinned_src),
                     vectors);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(FKV_ERR_RUNTIME, "plan upload launch failed: %s", hipGetErrorString(e));
  return FKV_OK;
}

int common_vector_width(const uint64_t *vals, int n) {
  uint64_t acc = 0;
  for (int i = 0; i < n; ++i)
    acc |= vals[i];
  for (int v = 16; v > 1; v >>= 1)
    if ((acc & (uint64_t)(v - 1)) == 0)
      return v;
  return 1;
}

namespace {
// Checks one job and fills in what the kernel derives from its shape; `total` = its
// work units (slices, or pieces in packed mode).  FKV_OK with *total == 0: nothing to do.
int prepare_job(CopyKernelArgs &a, int64_t *total, int *grid_pct) {
  *total = 0;
  *grid_pct = 100;
  if (a.num_blocks <= 0 || a.lk <= 0 || a.chunk_bytes <= 0)
    return FKV_OK;
  if (a.lk > kCopyMaxLK)
    return fail(FKV_ERR_RUNTIME, "copy kernel: %d (layer,kv) pairs exceed the LDS table (%d)",
                a.lk, kCopyMaxLK);
  if (a.vec != 16 && a.vec != 8 && a.vec != 4 && a.vec != 2 && a.vec != 1)
    return fail(FKV_ERR_RUNTIME, "copy kernel: bad vector width %d", a.vec);
  if (a.chunk_bytes % a.vec)
    return fail(FKV_ERR_RUNTIME, "copy kernel: chunk %lld not a multiple of vector width %d",
                (long long)a.chunk_bytes, a.vec);
  // Launches that HBM bounds (their callers ask for an unroll) go by the slice where the
  // chunks are at least as long as one; 16 vectors per lane for chunks of whole slices of that
  // size, if asked for.
  a.per_slice = a.unroll != 0 && a.vec == 16 && a.nt_store && !a.claim &&
                a.chunk_bytes >= (int64_t)kWave * kCopyUnroll * 16;
  if (!(a.per_slice && a.unroll == kCopyUnrollDeep &&
        a.chunk_bytes % ((int64_t)kWave * kCopyUnrollDeep * 16) == 0))
    a.unroll = kCopyUnroll;
  const int64_t slice_bytes = (int64_t)kWave * a.unroll * a.vec;
  const int64_t slices = (a.chunk_bytes + slice_bytes - 1) / slice_bytes;
  const int64_t spp = slices * a.lk;
  // The kernel indexes slices inside an id tile with 32 bits.
  if (slices > INT32_MAX || spp * kCopyIdTile > (int64_t)UINT32_MAX)
    return fail(FKV_ERR_RUNTIME,
                "copy kernel: chunk of %lld B x %d (layer,kv) pairs is too large for one launch",
                (long long)a.chunk_bytes, a.lk);
  a.slices_per_chunk = (int32_t)slices;
  *total = spp * a.num_blocks;
  // Chunks that are no whole number of slices would leave lanes of a wavefront idle and requests
  // of it unissued in their last slice: they are packed (the kernel indexes vectors inside an
  // id tile with 32 bits).  48 MiB, us, short last slices (and as many more workgroups) -> packed:
  // host->GPU chunks of 9 KiB 951 -> 919, 18 KiB 921 -> 918; GPU->host 22 224 bytes 939 -> 930,
  // 64 KiB less a vector 936 -> 925; 1 MiB the same or 1 us less.  Launches that HBM bounds stay
  // with slices where a chunk has one.
  const int64_t vpp = a.chunk_bytes / a.vec * a.lk;
  a.packed = (a.chunk_bytes % slice_bytes != 0 && !a.per_slice && vpp * kCopyIdTile <= (int64_t)UINT32_MAX) ? 1 : 0;
  if (a.packed) {
    const int64_t piece = (int64_t)kWave * a.unroll;
    *total = (vpp * a.num_blocks + piece - 1) / piece;
    if (a.packed_grid_pct > 0)
      *grid_pct = a.packed_grid_pct;
  } else {
    // Too large to be packed: a wavefront has one slice in flight, and the last slice of a chunk
    // may be short.  As many workgroups more make up for it.
    *grid_pct = (int)((slices * slice_bytes * 100 + a.chunk_bytes - 1) / a.chunk_bytes);
  }
  return FKV_OK;
}

// Grid, workgroup size, mask and claims of a launch with `total` work units and
// `bytes` to move; `a` is the (first) job, whose mask, counters and choices count.
void shape_launch(CopyKernelArgs &a, int64_t total, int64_t bytes, int grid_pct,
                  int num_workgroups, int threads_per_workgroup, int64_t *grid_out,
                  int *threads_out) {
  int threads = threads_per_workgroup;
  if (threads < kWave)
    threads = kWave;
  if (threads > kCopyBlockThreads)
    threads = kCopyBlockThreads;
  threads = threads / kWave * kWave;
  const int waves_per_wg = threads / kWave;
  int64_t grid = num_workgroups > 0 ? num_workgroups : 1;
  if (grid_pct > 100)
    grid = (grid * grid_pct + 99) / 100;
  const int64_t useful = (total + waves_per_wg - 1) / waves_per_wg;
  if (grid > useful)
    grid = useful;
  if (grid < 1)
    grid = 1;
  // 0 = every XCD; a mask needs claim counters and must leave some XCD of the device out
  const uint32_t present = a.xcd_present ? a.xcd_present : 0xffu;
  if (!a.claim || (a.xcd_mask & present) == present)
    a.xcd_mask = 0;
  if (a.safety_net_wait_us <= 0)
    a.safety_net_wait_us = 50;
  a.num_claims = 0;
  // a number for this launch that no counter can hold by accident for long: counters
  // are zero at first, and 2^32 - 1 launches pass before a number comes back
  static std::atomic<uint32_t> launches{0};
  do {
    a.epoch = launches.fetch_add(1, std::memory_order_relaxed) + 1;
  } while (a.epoch == 0);
  if (a.xcd_mask != 0) {
    // `claims_per_wg` ranges per working workgroup (the caller's choice, 1 if it
    // makes none); `grid` working workgroups need grid / (selected XCDs) rounds over
    // all XCDs of the device.
    const int per_wg = a.claims_per_wg > 0 ? a.claims_per_wg : 1;
    a.num_claims = (uint32_t)std::min<int64_t>(grid * per_wg, total);
    const int per_round = std::max(1, __builtin_popcount(a.xcd_mask & present));
    grid = (grid + per_round - 1) / per_round * __builtin_popcount(present);
  } else if (a.claim && a.claims_per_wg > 0) {
    // All XCDs, some of which may be busy with the other direction (a transfer of
    // another stream or process that started later).  With several ranges per
    // workgroup (all_claims_per_wg of the launch policy, e.g. 8) the workgroups there
    // take fewer of them:
    // a restore that stays on all XCDs next to a put loop moves 23-24 instead of
    // 16-17 GB/s.  Off by default: alone, the same restore loses 2 % to the claims.
    const int per_wg = a.claims_per_wg;
    // ranges of 128 KiB at least: a claim costs a round trip to device memory
    a.num_claims = (uint32_t)std::min<int64_t>(std::min<int64_t>(grid * per_wg, total),
                                                bytes / (128 * 1024));
    if (a.num_claims <= (uint32_t)grid) // nothing to hand out: fixed shares
      a.num_claims = 0;
  }
  if (a.report)
    a.report->claims = a.report->claims || a.num_claims != 0;
  stats().kernel_launches.fetch_add(1, std::memory_order_relaxed);
  if (a.xcd_mask != 0)
    stats().confined_launches.fetch_add(1, std::memory_order_relaxed);
  *grid_out = grid;
  *threads_out = threads;
}

// Puts the tables of all jobs, lists that several of them share once, into the arguments of their
// launch; false (and nothing changed) where they do not fit.
bool jobs_into_arguments(CopyJobs &t, ArgPlan &plan) {
  CopyKernelArgs packed[kCopyMaxJobs];
  int words = 0;
  for (int j = 0; j < t.njobs; ++j) {
    packed[j] = t.job[j];
    if (!into_arguments(packed[j], packed, j, plan, &words))
      return false;
  }
  std::copy(packed, packed + t.njobs, t.job);
  return true;
}

template <int VEC>
int launch_jobs_vec(CopyJobs &t, int grid, int threads, size_t lds_bytes, hipStream_t stream) {
  ArgPlan plan;
  if (t.job[0].done.used)
    *t.job[0].done.used = true;
  if (VEC == 16 && jobs_into_arguments(t, plan)) {
    if (t.job[0].report)
      t.job[0].report->in_arguments = true;
    if (t.job[0].nt_store)
      hipLaunchKernelGGL((fkv_copy_jobs_args_kernel<true, false>), dim3(grid), dim3(threads), lds_bytes,
                         stream, t, plan);
    else if (t.job[0].lane_runs)
      hipLaunchKernelGGL((fkv_copy_jobs_args_kernel<false, true>), dim3(grid), dim3(threads), lds_bytes,
                         stream, t, plan);
    else
      hipLaunchKernelGGL((fkv_copy_jobs_args_kernel<false, false>), dim3(grid), dim3(threads), lds_bytes,
                         stream, t, plan);
  } else if (t.job[0].nt_store)
    hipLaunchKernelGGL((fkv_copy_jobs_kernel<VEC, true, kCopyUnroll>), dim3(grid), dim3(threads),
                       lds_bytes, stream, t);
  else if (VEC == 16 && t.job[0].lane_runs)
    hipLaunchKernelGGL((fkv_copy_jobs_kernel<16, false, kCopyUnroll, true>), dim3(grid),
                       dim3(threads), lds_bytes, stream, t);
  else
    hipLaunchKernelGGL((fkv_copy_jobs_kernel<VEC, false, kCopyUnroll>), dim3(grid), dim3(threads),
                       lds_bytes, stream, t);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(FKV_ERR_RUNTIME, "copy kernel launch failed: %s", hipGetErrorString(e));
  if (t.job[0].report)
    t.job[0].report->announced = t.job[0].done.word != nullptr;
  return FKV_OK;
}
} // namespace

int launch_copy_kernel(CopyKernelArgs a, int num_workgroups, int threads_per_workgroup,
                       hipStream_t stream) {
  int64_t total = 0;
  int grid_pct = 100;
  const bool hbm_bound = a.unroll != 0;
  FKV_TRY(prepare_job(a, &total, &grid_pct));
  if (total == 0)
    return FKV_OK;
  int64_t grid = 1;
  int threads = kWave;
  if (hbm_bound && threads_per_workgroup > kSliceWgThreads) {
    // the same number of wavefronts in smaller workgroups, which find room on a CU sooner (packed,
    // 1024 -> 256 lanes: 146 MiB out of chunks of 2880 bytes 83 -> 76 us, 60 MiB of 2304 54 -> 51,
    // 80 MiB of 4 KiB 57 -> 52)
    num_workgroups = (int)std::min<int64_t>(
        (int64_t)num_workgroups * threads_per_workgroup / kSliceWgThreads, INT32_MAX);
    threads_per_workgroup = kSliceWgThreads;
  }
  shape_launch(a, total, (int64_t)a.num_blocks * a.lk * a.chunk_bytes, grid_pct,
               num_workgroups, threads_per_workgroup, &grid, &threads);
  const size_t lds_bytes =
      !a.per_slice ? (size_t)(2 * a.lk + 2 * kCopyIdTile) * sizeof(uint64_t)
      : (int64_t)a.num_blocks * a.lk * a.chunk_bytes >= kSliceFewWgBytes ? kSliceLdsBytes
                                                                         : 0;
  switch (a.vec) {
  case 16: return launch_vec<16>(a, (int)grid, threads, lds_bytes, stream);
  case 8:  return launch_vec<8>(a, (int)grid, threads, lds_bytes, stream);
  case 4:  return launch_vec<4>(a, (int)grid, threads, lds_bytes, stream);
  case 2:  return launch_vec<2>(a, (int)grid, threads, lds_bytes, stream);
  default: return launch_vec<1>(a, (int)grid, threads, lds_bytes, stream);
  }
}

int launch_copy_jobs(const CopyKernelArgs *jobs, int njobs, int num_workgroups,
                     int threads_per_workgroup, hipStream_t stream) {
  if (njobs < 1 || njobs > kCopyMaxJobs)
    return fail(FKV_ERR_RUNTIME, "copy kernel: %d jobs in one launch (1..%d)", njobs, kCopyMaxJobs);
  CopyJobs t{};
  int64_t total = 0, bytes = 0;
  int max_lk = 0;
  int grid_pct = 100; // the largest any job asks for
  for (int j = 0; j < njobs; ++j) {
    CopyKernelArgs a = jobs[j];
    a.unroll = 0;
    a.lane_runs = jobs[0].lane_runs; // the launch's choice, made for the first job
    if (a.vec != jobs[0].vec || a.nt_store != jobs[0].nt_store)
      return fail(FKV_ERR_RUNTIME, "copy kernel: jobs of one launch differ in vector width or store kind");
    int64_t job_total = 0;
    int job_pct = 100;
    FKV_TRY(prepare_job(a, &job_total, &job_pct));
    if (job_total == 0)
      continue;
    const int64_t job_bytes = (int64_t)a.num_blocks * a.lk * a.chunk_bytes;
    // the line is measured in 4 KiB, so that units x weight stays far from 64 bits
    t.weight[t.njobs] = (uint32_t)std::max<int64_t>(1, std::min<int64_t>(job_bytes >> 12, UINT32_MAX));
    t.job[t.njobs++] = a;
    total += job_total;
    bytes += job_bytes;
    max_lk = std::max(max_lk, (int)a.lk);
    grid_pct = std::max(grid_pct, job_pct);
  }
  if (t.njobs == 0)
    return FKV_OK;
  // mask, counters and ranges per workgroup are those of the first job given
  t.job[0].xcd_mask = jobs[0].xcd_mask;
  t.job[0].claim = jobs[0].claim;
  t.job[0].claims_per_wg = jobs[0].claims_per_wg;
  t.job[0].xcd_present = jobs[0].xcd_present;
  t.job[0].safety_net_wait_us = jobs[0].safety_net_wait_us;
  t.job[0].packed_grid_pct = jobs[0].packed_grid_pct;
  t.job[0].report = jobs[0].report;
  t.job[0].done = jobs[0].done;
  int64_t grid = 1;
  int threads = kWave;
  shape_launch(t.job[0], total, bytes, grid_pct, num_workgroups, threads_per_workgroup, &grid,
               &threads);
  const size_t lds_bytes = (size_t)(2 * max_lk + 2 * kCopyIdTile) * sizeof(uint64_t);
  switch (t.job[0].vec) {
  case 16: return launch_jobs_vec<16>(t, (int)grid, threads, lds_bytes, stream);
  case 8:  return launch_jobs_vec<8>(t, (int)grid, threads, lds_bytes, stream);
  case 4:  return launch_jobs_vec<4>(t, (int)grid, threads, lds_bytes, stream);
  case 2:  return launch_jobs_vec<2>(t, (int)grid, threads, lds_bytes, stream);
  default: return launch_jobs_vec<1>(t, (int)grid, threads, lds_bytes, stream);
  }
}

namespace {
// A layerwise restore in one launch: every batch of layers, in order, announced as it lands.
//
// A launch a batch is bound by what lies around the launches: 8 us between two of them on a
// stream, a ramp and a tail each, and 20 us of host time for a launch, its event and the
// consumer's wait, next to 5 us (256 KiB) to 18 us (1 MiB) of link time.  Here the wavefronts
// claim ranges of 128 KiB that run through all batches, so the link never drains between two
// of them, and a batch costs the host nothing.
//
// A batch has landed when all its ranges are counted.  A range is counted behind a release
// fence, which also waits for its stores; that, the answer of the counter and the next claim
// are looked at when the first vectors of the following range have arrived, a round trip over
// the link later, when they have long come back.  (Counted right behind its stores, with the
// claim read through LDS, a range cost the wavefront 3 us more: 8 % of 32 layers of 1 MiB with 16
// wavefronts.)  Write-through stores instead of the fence were 5 % slower with 24 wavefronts.  Whoever counts the last range of a batch
// writes its epoch to a word in device memory, which streams wait for, and one in pinned
// memory, which the host looks at (see Landing).
//
// Whole restores, the forward stream waiting for every layer (us, a launch a batch -> this):
// 8 x 256 KiB to eventfds 159 -> 72, 32 x 1 MiB 773 -> 627, 61 x 7 MiB 9190 (rows gathered by host threads)
// -> 7631, which is 56.6 GB/s.  Next to a fused attention of 76 us a layer: 32 x 1 MiB 2845 -> 2807,
// 61 x 7 MiB 9193 -> 7855; next to three 2048^3 GEMMs a layer: 2691 -> 2561, 9224 -> 8044.
// Chunks of no whole number of slices are packed, batch by batch, as in copy_share: a batch is a
// sequence of vectors, position-major, cut into pieces of a slice.  Short chunks used to take a
// launch a batch (us, before -> this): 55 x 122 KiB in chunks of 2304 bytes 618 -> 170, 31 x 824 KiB
// 946 -> 521; 8 batches of 5 chunks, a stream waiting for each, 149 -> 58.  Longer ones had short last
// slices: 41 x 4.6 MiB in chunks of 18 KiB 3567 -> 3502, 61 x 1.1 MiB 1326 -> 1324.
template <bool PACKED>
__device__ __forceinline__ void copy_layers(const LayersLaunch &t, const CopyKernelArgs &a) {
  using V = VecType<16>::type;
  __shared__ uint64_t s_base_src[kCopyMaxLK], s_base_dst[kCopyMaxLK];
  __shared__ int64_t s_off_src[kCopyIdTile], s_off_dst[kCopyIdTile];
  __shared__ uint32_t s_claim;
  Shares shares(a);
  if (!shares.enter(&s_claim))
    return;
  const int lane = threadIdx.x;
  constexpr int64_t kSliceBytes = (int64_t)kWave * kCopyUnroll * 16;
  constexpr uint32_t kPiece = kWave * kCopyUnroll;
  const uint32_t slices = (uint32_t)a.slices_per_chunk;
  const uint32_t vpc = (uint32_t)(a.chunk_bytes / 16);
  const uint32_t q64 = kWave / vpc, r64 = kWave % vpc; // 64 vectors = q64 chunks + r64
  uint32_t tile = 0; // first of the block positions whose offsets are in LDS
  auto load_tile = [&](uint32_t at) {
    __syncthreads();
    const uint32_t n = min((uint32_t)kCopyIdTile, (uint32_t)a.num_blocks - at);
    for (uint32_t i = lane; i < n; i += kWave) {
      s_off_src[i] = a.ids_src[at + i] * a.stride_src;
      s_off_dst[i] = a.ids_dst[at + i] * a.stride_dst;
    }
    __syncthreads();
    tile = at;
  };
  for (int i = lane; i < a.lk; i += kWave) {
    s_base_src[i] = a.base_src[i];
    s_base_dst[i] = a.base_dst[i];
  }
  load_tile(0);

  Landing landing(t, lane == 0);
  // The claim after the current one; a safety-net workgroup claims none ahead of time.
  auto claim_ahead = [&]() -> uint32_t {
    const uint32_t c = from_first_lane(shares.next_claim);
    if (lane == 0 && c < a.num_claims)
      shares.next_claim = shares.claim_one();
    return c;
  };
  auto claim_now = [&]() -> uint32_t {
    uint32_t c, all;
    return shares.next(&s_claim, &c, &all) ? c : a.num_claims;
  };
  uint32_t part = shares.safety_net ? claim_now() : claim_ahead();
  while (part < a.num_claims) {
    uint32_t ahead = a.num_claims;
    const uint32_t batch = part / (uint32_t)t.ranges, range = part - batch * (uint32_t)t.ranges;
    const uint32_t ranges = t.ranges_of((int)batch);
    const uint32_t pair0 = batch * (uint32_t)t.pairs_per_batch;
    const uint32_t pairs = min((uint32_t)t.pairs_per_batch, (uint32_t)a.lk - pair0);
    const uint32_t spp = pairs * (PACKED ? vpc : slices);
    const uint32_t vectors = (uint32_t)a.num_blocks * spp; // packed: checked on the host
    const uint64_t units = PACKED ? (vectors + kPiece - 1) / kPiece : (uint64_t)a.num_blocks * spp;
    const uint64_t s0 = units * range / ranges;
    const uint64_t s1 = units * (range + 1) / ranges;
    const uint32_t qlk = q64 / pairs, rlk = q64 - qlk * pairs; // q64 chunks = qlk positions + rlk
    for (uint64_t s = s0; s < s1; ++s) {
      const V *src[kCopyUnroll];
      V *dst[kCopyUnroll];
      int nvec; // vectors of the piece: those of a lane are 64 apart
      if (PACKED) {
        const uint32_t v0 = (uint32_t)s * kPiece, last = min(v0 + kPiece, vectors) - 1;
        const uint32_t first_p = v0 / spp, last_p = last / spp;
        if (first_p < tile || last_p - tile >= (uint32_t)kCopyIdTile)
          load_tile(first_p); // a piece spans 512 positions at most
        nvec = (int)(last + 1 - v0);
        // located by division, the further ones by adding quotients and remainders; lanes
        // beyond the end stay on their last valid vector
        uint32_t v = v0 + lane;
        const uint32_t vc = min(v, last);
        const uint32_t c = vc / vpc;
        uint32_t w = vc - c * vpc, p = c / pairs, i = c - p * pairs;
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) {
          if (u > 0) {
            v += kWave;
            uint32_t w2 = w + r64, i2 = i + rlk, p2 = p + qlk;
            if (w2 >= vpc) {
              w2 -= vpc;
              i2 += 1;
            }
            if (i2 >= pairs) {
              i2 -= pairs;
              p2 += 1;
            }
            const bool ok = v <= last;
            w = ok ? w2 : w;
            i = ok ? i2 : i;
            p = ok ? p2 : p;
          }
          src[u] = reinterpret_cast<const V *>(s_base_src[pair0 + i] + (uint64_t)s_off_src[p - tile]) + w;
          dst[u] = reinterpret_cast<V *>(s_base_dst[pair0 + i] + (uint64_t)s_off_dst[p - tile]) + w;
        }
      } else {
        const uint32_t p = (uint32_t)(s / spp);
        const uint32_t r = (uint32_t)(s - (uint64_t)p * spp);
        const uint32_t i = r / slices, sl = r - i * slices;
        if (p - tile >= (uint32_t)kCopyIdTile) // behind the tile, or before it (wraps)
          load_tile(p / kCopyIdTile * kCopyIdTile);
        const int64_t off = (int64_t)sl * kSliceBytes;
        const int64_t left = a.chunk_bytes - off;
        nvec = (int)((left < kSliceBytes ? left : kSliceBytes) / 16);
        const V *from = reinterpret_cast<const V *>(s_base_src[pair0 + i] +
                                                    (uint64_t)s_off_src[p - tile] + off);
        V *to = reinterpret_cast<V *>(s_base_dst[pair0 + i] + (uint64_t)s_off_dst[p - tile] + off);
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) {
          src[u] = from + min(u * kWave + lane, nvec - 1);
          dst[u] = to + u * kWave + lane;
        }
      }
      V v[kCopyUnroll];
#pragma unroll
      for (int u = 0; u < kCopyUnroll; ++u)
        v[u] = get<V, true>(src[u]);
      // The vectors come from the other end of the link, so by the time they are here every
      // store of the range before has completed, and the answers of the two counters have come:
      // nothing is waited for that is not there.
      if (s == s0 || landing.counted >= 0)
        drain_wave();
      landing.announce();
      if (s == s0) {
        if (landing.copied >= 0)
          landing.count();
        if (!shares.safety_net)
          ahead = claim_ahead();
      }
      if (nvec == (int)kPiece) {
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u)
          put<V, true>(v[u], dst[u]);
      } else {
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u)
          if (u * kWave + lane < nvec)
            put<V, true>(v[u], dst[u]);
        nothing_in_flight();
      }
    }
    landing.copied = (int)batch;
    part = shares.safety_net ? claim_now() : ahead;
  }
  drain_wave();
  landing.announce();
  if (landing.copied >= 0)
    landing.count();
  landing.announce();
}
template <bool PACKED> __global__ __launch_bounds__(kWave) void fkv_copy_layers_kernel(LayersLaunch t) {
  copy_layers<PACKED>(t, t.a);
}
template <bool PACKED>
__global__ __launch_bounds__(kWave) void fkv_copy_layers_args_kernel(LayersLaunch t, ArgPlan plan) {
  CopyKernelArgs a = t.a;
  tables_from_arguments(a, plan);
  copy_layers<PACKED>(t, a);
}

// Holds its stream until batches have landed, as an event behind them would: for as long as that
// takes.  The launch it waits for was submitted before it, but may lie behind other work of its
// hardware queue for any length of time (a collective that waits for another rank), so no clock
// ends the wait; the host does, should it find that the launch ended in an error.  One
// wavefront, a word a lane: the words are written in any order.
__global__ __launch_bounds__(kWave) void fkv_wait_landed_kernel(const uint64_t *landed, uint32_t count,
                                                                uint64_t epoch,
                                                                const uint64_t *given_up) {
  uint32_t looks = 0;
  // relaxed: what the stream runs next starts with an acquire of its own
  for (uint32_t i = threadIdx.x; i < count; i += kWave)
    while (__hip_atomic_load(landed + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) < epoch) {
      // that word lies at the other end of the link: every 0.1 ms or so
      if (++looks % 64 == 0 &&
          __hip_atomic_load(given_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) >= epoch)
        return;
      __builtin_amdgcn_s_sleep(8);
    }
}

int launch_layers(LayersLaunch t, int num_workgroups, hipStream_t stream) {
  int64_t total = 0;
  int grid_pct = 100;
  FKV_TRY(prepare_job(t.a, &total, &grid_pct));
  // vectors of a batch, which the kernel counts in 32 bits
  const int64_t vpb = t.a.chunk_bytes / 16 * t.pairs_per_batch * t.a.num_blocks;
  if (total == 0 || t.a.vec != 16 || !t.a.claim || t.batches < 1 ||
      (t.a.packed && vpb > kLayersMaxVectors))
    return fail(FKV_ERR_RUNTIME, "copy kernel: a restore of this shape has no single launch");
  int64_t grid = 1;
  int threads = kWave;
  shape_launch(t.a, total, (int64_t)t.a.num_blocks * t.a.lk * t.a.chunk_bytes,
               grid_pct * t.grid_pct / 100, num_workgroups, kWave, &grid, &threads);
  const uint32_t present = t.a.xcd_present ? t.a.xcd_present : 0xffu;
  const int64_t working =
      t.a.xcd_mask ? grid * __builtin_popcount(t.a.xcd_mask & present) /
                         std::max(1, __builtin_popcount(present))
                   : grid;
  const int64_t last_pairs = t.a.lk - (int64_t)(t.batches - 1) * t.pairs_per_batch;
  constexpr int64_t kPiece = kWave * kCopyUnroll;
  const int64_t vectors = t.a.chunk_bytes / 16 * t.a.num_blocks; // of a pair
  LayersCut cut = cut_layers(t.batches, t.pairs_per_batch, last_pairs,
                             t.a.packed ? std::max<int64_t>(1, vectors / kPiece)
                                        : (int64_t)t.a.num_blocks * t.a.slices_per_chunk, working);
  if (t.a.packed) { // none empty
    cut.ranges = std::min(cut.ranges, (vectors * t.pairs_per_batch + kPiece - 1) / kPiece);
    cut.last_ranges = std::min({cut.last_ranges, cut.ranges, (vectors * last_pairs + kPiece - 1) / kPiece});
  }
  if (last_pairs < 1 || cut.claims(t.batches) > (int64_t)INT32_MAX)
    return fail(FKV_ERR_RUNTIME, "copy kernel: %d batches of %d of %d (layer, kv) pairs", t.batches,
                t.pairs_per_batch, t.a.lk);
  t.ranges = (int32_t)cut.ranges;
  t.last_ranges = (int32_t)cut.last_ranges;
  t.a.num_claims = (uint32_t)cut.claims(t.batches);
  LayersLaunch with_plan = t;
  ArgPlan plan;
  int words = 0;
  if (into_arguments(with_plan.a, nullptr, 0, plan, &words)) {
    hipLaunchKernelGGL(t.a.packed ? fkv_copy_layers_args_kernel<true> : fkv_copy_layers_args_kernel<false>,
                       dim3((unsigned)grid), dim3(kWave), 0, stream, with_plan, plan);
  } else {
    hipLaunchKernelGGL(t.a.packed ? fkv_copy_layers_kernel<true> : fkv_copy_layers_kernel<false>,
                       dim3((unsigned)grid), dim3(kWave), 0, stream, t);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(FKV_ERR_RUNTIME, "copy kernel launch failed: %s", hipGetErrorString(e));
  return FKV_OK;
}

int wait_landed(const uint64_t *landed, const uint64_t *landed_host, int count, uint64_t epoch,
                const uint64_t *given_up, int device, hipEvent_t behind, hipStream_t stream) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {
    (void)hipGetLastError();
    capture = hipStreamCaptureStatusActive; // let the event decide
  }
  if (capture != hipStreamCaptureStatusNone) {
    FKV_HIP_TRY(hipStreamWaitEvent(stream, behind, 0));
    return FKV_OK;
  }
  int first = 0; // not known to have landed yet
  while (first < count && __atomic_load_n(landed_host + first, __ATOMIC_ACQUIRE) >= epoch)
    ++first;
  if (first == count)
    return FKV_OK; // they are there: whatever the stream gets next finds them
  // a consumer on another GPU looks at the words in host memory
  int of_stream = -1; // the null stream: that of the current device
  if (stream && hipStreamGetDevice(stream, &of_stream) != hipSuccess) {
    (void)hipGetLastError();
    of_stream = -1;
  }
  DeviceGuard guard(of_stream);
  if (!guard.ok())
    return fail(FKV_ERR_RUNTIME, "cannot select the device of the consumer's stream");
  const uint64_t *words = (guard.device() == device ? landed : landed_host) + first;
  FKV_LAUNCH_BESIDE(fkv_wait_landed_kernel, stream, words, (uint32_t)(count - first), epoch, given_up);
  FKV_HIP_TRY(hipGetLastError());
  return FKV_OK;
}

const LayersDevice kLayersDevice{launch_layers, wait_landed};
[[maybe_unused]] const bool layers_device_set = (layers_device = &kLayersDevice, true);
bool not_capturing(hipStream_t stream) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) == hipSuccess)
    return capture == hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return false;
}
[[maybe_unused]] const bool copies_announce_set = (copies_announce = not_capturing, true);
} // namespace

} // namespace fkv

// ---- what HBM delivers to a streaming kernel ---------------------------------
namespace fkv {
namespace {
typedef unsigned int hbm_vec __attribute__((ext_vector_type(4)));
// MODE 0: read only, 1: write only, 2: copy.  Contiguous memory, 16 vectors of 16
// bytes in flight per lane, nontemporal accesses, wavefronts take slices round-robin:
// the shape that measured fastest for all three.
template <int MODE>
__global__ __launch_bounds__(1024) void fkv_hbm_yardstick_kernel(const hbm_vec *__restrict__ src,
                                                                 hbm_vec *__restrict__ dst,
                                                                 size_t nvec, hbm_vec *sink) {
  constexpr int U = 16;
  const int lane = threadIdx.x & 63;
  const size_t wave = (size_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  const size_t nwaves = (size_t)gridDim.x * (blockDim.x / 64);
  const size_t slice = 64 * U;
  hbm_vec acc = {0, 0, 0, 0};
  for (size_t s = wave * slice; s + slice <= nvec; s += nwaves * slice) {
    hbm_vec r[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      r[u] = MODE == 1 ? hbm_vec{(unsigned)s, (unsigned)u, 3u, 4u}
                       : __builtin_nontemporal_load(src + s + u * 64 + lane);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (MODE == 0)
        acc ^= r[u];
      else
        __builtin_nontemporal_store(r[u], dst + s + u * 64 + lane);
    }
  }
  // never true for the fill pattern of the caller; keeps the loads of MODE 0 alive
  if (MODE == 0 && acc.x == 0x12345678u && acc.y == 0x9abcdef0u)
    *sink = acc;
}
} // namespace
} // namespace fkv

extern "C" int fkv_measure_hbm_rate(int32_t device, size_t bytes, int32_t reps, int32_t mode,
                                    double *best_gbps, double *median_gbps) try {
  using namespace fkv;
  clear_error();
  if (bytes < (1u << 20) || reps < 1 || mode < 0 || mode > 2 || !best_gbps)
    return fail(FKV_ERR_INVALID_ARG, "fkv_measure_hbm_rate: bad arguments");
  DeviceGuard guard(device);
  if (!guard.ok())
    return fail(FKV_ERR_RUNTIME, "cannot select HIP device %d", device);
  bytes &= ~(size_t)(64 * 16 * 16 - 1); // whole slices
  hbm_vec *src = nullptr, *dst = nullptr, *sink = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  std::vector<double> rates;
  int rc = FKV_OK;
  auto cleanup = [&] {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (src) (void)hipFree(src);
    if (dst) (void)hipFree(dst);
    if (sink) (void)hipFree(sink);
    (void)hipGetLastError();
  };
#define HB_TRY(x)                                                              \
  do {                                                                         \
    hipError_t e_ = (x);                                                       \
    if (e_ != hipSuccess) {                                                    \
      (void)hipGetLastError();                                                 \
      rc = fail(FKV_ERR_RUNTIME, "%s: %s", #x, hipGetErrorString(e_));         \
      cleanup();                                                               \
      return rc;                                                               \
    }                                                                          \
  } while (0)
  HB_TRY(hipMalloc(reinterpret_cast<void **>(&src), bytes));
  HB_TRY(hipMalloc(reinterpret_cast<void **>(&dst), bytes));
  HB_TRY(hipMalloc(reinterpret_cast<void **>(&sink), 64));
  HB_TRY(hipEventCreate(&e0));
  HB_TRY(hipEventCreate(&e1));
  HB_TRY(hipMemset(src, 0x11, bytes));
  HB_TRY(hipMemset(dst, 0x22, bytes));
  const size_t nvec = bytes / 16;
  for (int r = -1; r < reps; ++r) { // r == -1 is an untimed warm-up
    HB_TRY(hipEventRecord(e0, nullptr));
    if (mode == 0)
      hipLaunchKernelGGL(fkv_hbm_yardstick_kernel<0>, dim3(8192), dim3(1024), 0, nullptr, src, dst, nvec, sink);
    else if (mode == 1)
      hipLaunchKernelGGL(fkv_hbm_yardstick_kernel<1>, dim3(8192), dim3(1024), 0, nullptr, src, dst, nvec, sink);
    else
      hipLaunchKernelGGL(fkv_hbm_yardstick_kernel<2>, dim3(8192), dim3(1024), 0, nullptr, src, dst, nvec, sink);
    HB_TRY(hipGetLastError());
    HB_TRY(hipEventRecord(e1, nullptr));
    HB_TRY(hipEventSynchronize(e1));
    float ms = 0;
    HB_TRY(hipEventElapsedTime(&ms, e0, e1));
    if (r >= 0 && ms > 0)
      rates.push_back((mode == 2 ? 2.0 : 1.0) * (double)bytes / (ms * 1e-3) / 1e9);
  }
#undef HB_TRY
  cleanup();
  if (rates.empty())
    return fail(FKV_ERR_RUNTIME, "no timed repetition");
  std::sort(rates.begin(), rates.end());
  *best_gbps = rates.back();
  if (median_gbps)
    *median_gbps = rates[rates.size() / 2];
  return FKV_OK;
} catch (...) {
  return fkv::caught(__func__);
}

extern "C" int fkv_streams_run_concurrently(int32_t device, void *stream_a, void *stream_b,
                                            int32_t *concurrent) try {
  using namespace fkv;
  clear_error();
  if (!concurrent)
    return fail(FKV_ERR_INVALID_ARG, "fkv_streams_run_concurrently: null result pointer");
  DeviceGuard guard(device);
  if (!guard.ok())
    return fail(FKV_ERR_RUNTIME, "cannot select HIP device %d", device);
  hipStream_t a = static_cast<hipStream_t>(stream_a), b = static_cast<hipStream_t>(stream_b);
  if (a == b) {
    *concurrent = 0;
    return FKV_OK;
  }
  constexpr long long kTicks = 30000; // 0.3 ms
  auto timed = [&](bool both, double *ms) -> int {
    FKV_HIP_TRY(hipStreamSynchronize(a));
    FKV_HIP_TRY(hipStreamSynchronize(b));
    const auto t0 = std::chrono::steady_clock::now();
    hipLaunchKernelGGL(fkv_wait_kernel, dim3(1), dim3(64), 0, a, kTicks, nullptr);
    if (both)
      hipLaunchKernelGGL(fkv_wait_kernel, dim3(1), dim3(64), 0, b, kTicks, nullptr);
    FKV_HIP_TRY(hipGetLastError());
    FKV_HIP_TRY(hipStreamSynchronize(a));
    FKV_HIP_TRY(hipStreamSynchronize(b));
    *ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return FKV_OK;
  };
  double warm = 0, one = 1e30, two = 1e30;
  FKV_TRY(timed(true, &warm)); // first launches carry code-object loading
  for (int r = 0; r < 3; ++r) {
    double m = 0;
    FKV_TRY(timed(false, &m));
    one = std::min(one, m);
    FKV_TRY(timed(true, &m));
    two = std::min(two, m);
  }
  *concurrent = two < 1.5 * one ? 1 : 0;
  return FKV_OK;
} catch (...) {
  return fkv::caught(__func__);
}

extern "C" int fkv_streams_hand_over_us(int32_t device, void *stream_a, void *stream_b,
                                        double *round_trip_us) try {
  using namespace fkv;
  clear_error();
  if (!round_trip_us)
    return fail(FKV_ERR_INVALID_ARG, "fkv_streams_hand_over_us: null result pointer");
  DeviceGuard guard(device);
  if (!guard.ok())
    return fail(FKV_ERR_RUNTIME, "cannot select HIP device %d", device);
  hipStream_t a = static_cast<hipStream_t>(stream_a), b = static_cast<hipStream_t>(stream_b);
  constexpr int kRoundTrips = 16;
  constexpr long long kGateTicks = 200000; // 2 ms: the whole chain is enqueued before it may start
  hipEvent_t t0 = nullptr, t1 = nullptr, there[kRoundTrips] = {}, back[kRoundTrips] = {};
  auto cleanup = [&] {
    for (hipEvent_t e : {t0, t1})
      if (e)
        (void)hipEventDestroy(e);
    for (int k = 0; k < kRoundTrips; ++k)
      for (hipEvent_t e : {there[k], back[k]})
        if (e)
          (void)hipEventDestroy(e);
  };
#define HO_TRY(expr)                                                                      \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess) {                                                               \
      (void)hipStreamSynchronize(a);                                                      \
      (void)hipStreamSynchronize(b);                                                      \
      cleanup();                                                                          \
      (void)hipGetLastError();                                                            \
      return fail(FKV_ERR_RUNTIME, "fkv_streams_hand_over_us: %s", hipGetErrorString(e_)); \
    }                                                                                     \
  } while (0)
  HO_TRY(hipEventCreate(&t0));
  HO_TRY(hipEventCreate(&t1));
  for (int k = 0; k < kRoundTrips; ++k) {
    HO_TRY(hipEventCreateWithFlags(&there[k], kBookkeepingEvent));
    HO_TRY(hipEventCreateWithFlags(&back[k], kBookkeepingEvent));
  }
  double best = 1e30;
  for (int rep = 0; rep < 2; ++rep) { // the first one carries whatever is set up on first use
    HO_TRY(hipStreamSynchronize(a));
    HO_TRY(hipStreamSynchronize(b));
    hipLaunchKernelGGL(fkv_wait_kernel, dim3(1), dim3(64), 0, a, kGateTicks, nullptr);
    HO_TRY(hipGetLastError());
    HO_TRY(hipEventRecord(t0, a));
    for (int k = 0; k < kRoundTrips; ++k) {
      hipLaunchKernelGGL(fkv_wait_kernel, dim3(1), dim3(64), 0, a, 0ll, nullptr);
      HO_TRY(hipEventRecord(there[k], a));
      HO_TRY(hipStreamWaitEvent(b, there[k], 0));
      hipLaunchKernelGGL(fkv_wait_kernel, dim3(1), dim3(64), 0, b, 0ll, nullptr);
      HO_TRY(hipEventRecord(back[k], b));
      HO_TRY(hipStreamWaitEvent(a, back[k], 0));
    }
    HO_TRY(hipGetLastError());
    HO_TRY(hipEventRecord(t1, a));
    HO_TRY(hipEventSynchronize(t1));
    HO_TRY(hipStreamSynchronize(b));
    float ms = 0;
    HO_TRY(hipEventElapsedTime(&ms, t0, t1));
    best = std::min(best, (double)ms * 1e3 / kRoundTrips);
  }
#undef HO_TRY
  cleanup();
  *round_trip_us = best;
  return FKV_OK;
} catch (...) {
  return fkv::caught(__func__);
}
