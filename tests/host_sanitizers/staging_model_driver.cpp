// Payload transfers (fkv_staging_transfer) with the kernel on the CPU device model, for sanitizer
// builds: seeded calls over slots that are and are not multiples of a vector, payloads from nothing
// to the whole slot (ends of every number of vectors and bytes), sizes that do not fit, up to the
// largest 64 bits hold, split batches, both directions, both orders of vectors, against the oracle byte for byte.  Staging
// buffer, host cache, sizes and size table are allocations of exactly the size the call may touch.
#include <hip/hip_runtime.h>

#include "fkv_transfer.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <random>
#include <vector>

#define REQUIRE(cond, ...)                                                                          \
  do {                                                                                              \
    if (!(cond)) {                                                                                  \
      fprintf(stderr, "staging_model_driver: " __VA_ARGS__);                                        \
      fprintf(stderr, " [%s:%d]\n", __FILE__, __LINE__);                                            \
      exit(1);                                                                                      \
    }                                                                                               \
  } while (0)

extern "C" void fkv_oracle_staging_transfer(uint8_t *staging, int64_t staging_stride, uint64_t *comp_sizes,
                                            uint8_t *cpu, int64_t chunk_capacity, int32_t *overflow,
                                            int64_t cpu_kv_stride, int64_t cpu_layer_stride,
                                            int64_t cpu_block_stride, const int64_t *cpu_ids,
                                            uint32_t *size_table, int64_t table_block_stride,
                                            int64_t table_layer_stride, int start_layer, int kv_dim,
                                            int num_blocks, int batch_start, int bsz, int is_write_cpu);

namespace {

using Rng = std::mt19937_64;
int pick(Rng &rng, int lo, int hi) { return lo + (int)(rng() % (uint64_t)(hi - lo + 1)); }

template <typename T> T *memory(const std::vector<T> &v, bool pinned) {
  void *p = nullptr;
  const size_t bytes = v.size() * sizeof(T);
  REQUIRE((pinned ? hipHostMalloc(&p, bytes, 0) : hipMalloc(&p, bytes)) == hipSuccess, "memory");
  memcpy(p, v.data(), bytes);
  return static_cast<T *>(p);
}
template <typename T> bool same(const T *p, const std::vector<T> &v) {
  return memcmp(p, v.data(), v.size() * sizeof(T)) == 0;
}

// A size in [0, most]: often one at which a slice, a vector or nothing ends.
uint64_t size_up_to(Rng &rng, int64_t most) {
  const int64_t slice = 64 * 8 * 16;
  int64_t s = 0;
  switch (pick(rng, 0, 4)) {
  case 0: s = pick(rng, 0, 40); break;
  case 1: s = 16 * pick(rng, 0, 520) + (pick(rng, 0, 1) ? pick(rng, 0, 15) : 0); break;
  case 2: s = slice * pick(rng, 0, 3) + pick(rng, -17, 17); break;
  case 3: s = most - pick(rng, 0, 20); break;
  default: s = pick(rng, 0, 1 << 20) % (most + 1); break;
  }
  return (uint64_t)std::clamp<int64_t>(s, 0, most);
}
uint64_t too_large(Rng &rng, int64_t most, bool wide) {
  const std::vector<uint64_t> v = {(uint64_t)most + 1, (uint64_t)most + 4096, 0xffffffffu};
  const std::vector<uint64_t> w = {1ull << 32, (1ull << 32) + 16, 1ull << 63, (1ull << 63) + 100, 0ull - 1,
                                   0ull - 17, 0ull - 8191, 0ull - 8193, 0ull - (1ull << 33)};
  const size_t k = rng() % (v.size() + (wide ? w.size() : 0));
  return k < v.size() ? v[k] : w[k - v.size()];
}

void call(unsigned long long seed, hipStream_t stream) {
  Rng rng(seed);
  const bool write = rng() & 1, aligned = pick(rng, 0, 3) != 0;
  const int unit = aligned ? 16 : 1;
  const int64_t capacity = (int64_t)unit * pick(rng, 1, (pick(rng, 0, 2) ? 1200 : 60) * 16 / unit);
  const int64_t stride = capacity + unit * pick(rng, 0, 3);
  const int kv = pick(rng, 1, 2), blocks = pick(rng, 1, pick(rng, 0, 9) ? 12 : 500), pool = blocks + pick(rng, 0, 3),
            layers = pick(rng, 1, blocks > 12 ? 1 : 3), start_layer = pick(rng, 0, 2), all_layers = start_layer + layers;
  const int total = layers * kv * blocks, batch_start = pick(rng, 0, total - 1),
            bsz = std::min(total - batch_start, pick(rng, 0, 3) ? total : pick(rng, 1, 5));
  const bool block_first = rng() & 1;
  const int64_t kv_stride = block_first ? capacity : pool * capacity, layer_stride = kv * kv_stride,
                block_stride = block_first ? all_layers * kv * capacity : capacity;
  std::vector<uint8_t> staging(bsz * stride), host((size_t)all_layers * kv * pool * capacity);
  for (auto *v : {&staging, &host})
    for (auto &b : *v)
      b = (uint8_t)rng();
  std::vector<uint64_t> sizes(bsz, 99);
  std::vector<uint32_t> table((size_t)pool * all_layers * kv);
  for (auto &s : sizes)
    if (write)
      s = pick(rng, 0, 5) ? size_up_to(rng, capacity) : too_large(rng, capacity, true);
  for (auto &e : table)
    e = (uint32_t)(write || pick(rng, 0, 5) ? size_up_to(rng, capacity) : too_large(rng, stride, false));
  std::vector<int64_t> ids(pool);
  std::iota(ids.begin(), ids.end(), 0);
  std::shuffle(ids.begin(), ids.end(), rng);
  ids.resize(blocks);
  std::vector<int32_t> overflow = {3};
  const bool counted = write || (rng() & 1);

  uint8_t *d_staging = memory(staging, false), *h_host = memory(host, true);
  uint64_t *d_sizes = memory(sizes, false);
  uint32_t *h_table = memory(table, true);
  int32_t *d_overflow = memory(overflow, false);
  fkv_staging_transfer_desc d{};
  d.staging = d_staging, d.staging_stride = stride, d.comp_sizes = d_sizes, d.cpu_ptr = h_host;
  d.chunk_capacity = capacity, d.overflow = counted ? d_overflow : nullptr;
  d.cpu_kv_stride = kv_stride, d.cpu_layer_stride = layer_stride, d.cpu_block_stride = block_stride;
  d.cpu_block_ids = ids.data(), d.size_table = h_table;
  d.size_table_block_stride = all_layers * kv, d.size_table_layer_stride = kv;
  d.start_layer_id = start_layer, d.kv_dim = kv, d.num_blocks = blocks, d.batch_start = batch_start, d.bsz = bsz;
  d.is_write_cpu = write, d.transfer_num_cta = pick(rng, 0, 2), d.device = -1, d.sync = 1;
  fkv_launch_policy policy{}; // the order of vectors towards the host: not a number of `rng`, whose shapes stay
  REQUIRE(fkv_launch_policy_get(-1, &policy) == FKV_OK, "policy");
  policy.d2h_lane_runs = seed % 3 ? 2 : 0;
  REQUIRE(fkv_launch_policy_set(-1, &policy) == FKV_OK, "policy");
  REQUIRE(fkv_staging_transfer(&d, stream) == FKV_OK, "seed %llu: %s", seed, fkv_last_error());
  fkv_oracle_staging_transfer(staging.data(), stride, sizes.data(), host.data(), capacity,
                              counted ? overflow.data() : nullptr, kv_stride, layer_stride, block_stride,
                              ids.data(), table.data(), all_layers * kv, kv, start_layer, kv, blocks,
                              batch_start, bsz, write);
  REQUIRE(same(h_host, host), "seed %llu: host cache (write %d)", seed, write);
  REQUIRE(same(h_table, table), "seed %llu: size table (write %d)", seed, write);
  REQUIRE(same(d_staging, staging), "seed %llu: staging (write %d)", seed, write);
  REQUIRE(same(d_sizes, sizes), "seed %llu: sizes (write %d)", seed, write);
  REQUIRE(same(d_overflow, overflow), "seed %llu: overflow (write %d)", seed, write);
  REQUIRE(hipFree(d_staging) == hipSuccess && hipHostFree(h_host) == hipSuccess && hipFree(d_sizes) == hipSuccess &&
              hipHostFree(h_table) == hipSuccess && hipFree(d_overflow) == hipSuccess, "free");
}

} // namespace

int main(int argc, char **argv) {
  const int calls = argc > 1 ? atoi(argv[1]) : 100;
  hipStream_t stream = nullptr;
  REQUIRE(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) == hipSuccess, "stream");
  for (int i = 0; i < calls; ++i)
    call(70000 + i, stream);
  REQUIRE(hipStreamDestroy(stream) == hipSuccess, "stream");
  printf("ok: %d payload transfers\n", calls);
  return 0;
}
