// Layerwise restores that go out as one launch announcing its batches itself, over the
// emulated HIP runtime, for sanitizer builds: the words a launch announces its batches by and
// their reuse by later groups, consumers that wait for a word, both notify modes with
// eventfds, one and two GPUs, several groups at once, runtime calls refused part-way.  The
// launch is the stand-in of the emulated runtime, or the kernel itself on the CPU device model.
// Every byte is compared with a plain model.
#include <hip/hip_runtime_api.h>
#include <sys/eventfd.h>
#include <unistd.h>

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <random>
#include <thread>
#include <vector>

#include "fkv_transfer.h"

extern "C" {
long fkv_emulated_fail(int category, long after, long count); // emulated_hip_runtime.cpp
unsigned long long fkv_emulated_workgroups_run();
void fkv_emulated_hold_kernels(int on);
void fkv_emulated_clock_speed(long factor);
void fkv_emulated_kernel_tail(long us);
long fkv_emulated_host_waited_copies();
void fkv_emulated_late_words(long us);
}

#define REQUIRE(cond, ...)                                                                          \
  do {                                                                                              \
    if (!(cond)) {                                                                                  \
      fprintf(stderr, "FAILED %s:%d: %s\n  ", __FILE__, __LINE__, #cond);                           \
      fprintf(stderr, __VA_ARGS__);                                                                 \
      fprintf(stderr, "\n  last error: %s\n", fkv_last_error());                                    \
      _exit(1); /* kernels may be held: no destructor of the runtime could end */                   \
    }                                                                                               \
  } while (0)

namespace {

using Rng = std::mt19937_64;
int pick(Rng &rng, int lo, int hi) { return lo + (int)(rng() % (uint64_t)(hi - lo + 1)); }

void set_policy(int alt_kb = -1, int gather = 0) {
  for (int device = 0; device < 2; ++device) {
    fkv_launch_policy p{};
    REQUIRE(fkv_launch_policy_reset(device) == FKV_OK && fkv_launch_policy_get(device, &p) == FKV_OK,
            "policy");
    p.model_seed = 0;
    p.staged_restore = 0;
    p.staged_gather = gather;
    p.kernel_alt_stream_kb = alt_kb;
    REQUIRE(fkv_launch_policy_set(device, &p) == FKV_OK, "policy");
  }
}

uint64_t launches() {
  fkv_stats s{};
  fkv_get_stats(&s);
  return s.kernel_launches;
}

// Engine tensors per GPU and layer, [kv, pool, chunk], a block-first host pool, a group.
struct Group {
  int ranks, layers, kv, pool;
  int64_t chunk;
  std::vector<uint8_t *> dev; // [rank * layers + layer]
  std::vector<std::vector<uint8_t>> model;
  uint8_t *host = nullptr;
  std::vector<int32_t> fds;
  fkv_layerwise *g = nullptr;
  std::vector<int64_t> gids, cids;

  size_t layer_bytes() const { return (size_t)(kv * pool * chunk); }
  int64_t block() const { return layers * kv * chunk; }

  Group(Rng &rng, int ranks_, int layers_, int kv_, int pool_, int64_t chunk_)
      : ranks(ranks_), layers(layers_), kv(kv_), pool(pool_), chunk(chunk_) {
    std::vector<uint64_t> ptrs;
    for (int i = 0; i < ranks * layers; ++i) {
      uint8_t *d = nullptr;
      REQUIRE(hipMalloc((void **)&d, layer_bytes()) == hipSuccess, "engine tensor");
      memset(d, i, layer_bytes());
      dev.push_back(d);
      model.emplace_back(layer_bytes(), (uint8_t)i);
      ptrs.push_back((uint64_t)(uintptr_t)d);
      fds.push_back(eventfd(0, EFD_NONBLOCK));
    }
    REQUIRE(hipHostMalloc((void **)&host, (size_t)(pool * block()), 0) == hipSuccess, "host pool");
    std::vector<int64_t> kvs(ranks, pool * chunk), bs(ranks, chunk), ls(ranks, (int64_t)layer_bytes()),
        cs(ranks, chunk), devs;
    for (int r = 0; r < ranks; ++r)
      devs.push_back(r);
    fkv_layerwise_params p{};
    p.num_gpus = ranks;
    p.num_tensors_per_gpu = layers;
    p.gpu_block_ptrs_flat = ptrs.data();
    p.cpu_blocks_ptr = host;
    p.num_layers = layers;
    p.tp_size = ranks;
    p.gpu_kv_strides = kvs.data();
    p.gpu_block_strides = bs.data();
    p.gpu_layer_strides = ls.data();
    p.gpu_chunk_sizes = cs.data();
    p.gpu_device_ids = devs.data();
    p.layer_eventfds = fds.data();
    p.num_layer_eventfds = (int32_t)fds.size();
    fkv_ce_config_default(&p.ce);
    p.ce.is_blockfirst = 1;
    REQUIRE(fkv_layerwise_create(&p, &g) == FKV_OK, "create");
    refill(rng);
  }
  void refill(Rng &rng) { // new bytes in the host pool
    for (int64_t i = 0; i < pool * block(); i += 8) {
      const uint64_t v = rng();
      memcpy(host + i, &v, 8);
    }
  }
  int restore(Rng &rng, int n, int gran, int notify) {
    gids.resize(pool);
    cids.resize(pool);
    std::iota(gids.begin(), gids.end(), 0);
    std::iota(cids.begin(), cids.end(), 0);
    std::shuffle(gids.begin(), gids.end(), rng);
    std::shuffle(cids.begin(), cids.end(), rng);
    gids.resize(n);
    cids.resize(n);
    return fkv_layerwise_transfer(g, gids.data(), cids.data(), n, block(), chunk, kv * chunk, block(),
                                  4, 0, layers, gran, kv, 1, 0, "sharded", notify, 0);
  }
  void model_restore() {
    for (int r = 0; r < ranks; ++r)
      for (int l = 0; l < layers; ++l)
        for (int k = 0; k < kv; ++k)
          for (size_t q = 0; q < gids.size(); ++q)
            memcpy(model[r * layers + l].data() + (k * pool + gids[q]) * chunk,
                   host + cids[q] * block() + (l * kv + k) * chunk, (size_t)chunk);
  }
  void check(const char *when) {
    model_restore();
    for (size_t i = 0; i < dev.size(); ++i)
      REQUIRE(memcmp(dev[i], model[i].data(), layer_bytes()) == 0, "%s: tensor %zu differs", when, i);
  }
  int units(size_t i) {
    uint64_t v = 0;
    return read(fds[i], &v, 8) == 8 ? (int)v : 0;
  }
  void destroy() {
    fkv_layerwise_destroy(g);
    for (int fd : fds)
      close(fd);
    for (uint8_t *d : dev)
      REQUIRE(hipFree(d) == hipSuccess, "free");
    REQUIRE(hipHostFree(host) == hipSuccess, "free");
  }
};

int64_t some_chunk(Rng &rng) {
  return std::vector<int64_t>{8192, 8208, 18432, 8192 + 16 * pick(rng, 1, 700)}[pick(rng, 0, 3)];
}

// The words of a process's first group are set up without a copy on the null stream, which
// would wait for whatever the engine has queued there.
void first_words(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, 2, 3, 1, 2, 8192);
  set_policy(0); // plan memory and its counters: a restore of the same group, batch by batch
  REQUIRE(g.restore(rng, 2, 1, FKV_NOTIFY_HOSTFUNC) == FKV_OK, "restore");
  g.check("batch by batch");
  set_policy();
  const long before = fkv_emulated_host_waited_copies();
  REQUIRE(g.restore(rng, 2, 1, FKV_NOTIFY_HOSTFUNC) == FKV_OK, "restore");
  REQUIRE(fkv_emulated_host_waited_copies() == before, "%ld copies that wait for the null stream",
          fkv_emulated_host_waited_copies() - before);
  g.check("first words");
  g.destroy();
}

// Restores one after the other on one group, a consumer that waits for each layer.
void seeded_case(uint64_t seed) {
  Rng rng(seed);
  const int pool = pick(rng, 2, 7);
  Group g(rng, pick(rng, 1, 2), pick(rng, 2, 9), pick(rng, 1, 2), pool, some_chunk(rng));
  hipStream_t consumer = nullptr;
  REQUIRE(hipSetDevice(0) == hipSuccess &&
              hipStreamCreateWithFlags(&consumer, hipStreamNonBlocking) == hipSuccess, "stream");
  std::vector<std::vector<uint8_t>> seen(g.layers, std::vector<uint8_t>(g.layer_bytes()));
  for (int rep = 0; rep < 4; ++rep) {
    g.refill(rng);
    const int gran = pick(rng, 1, g.layers), batches = (g.layers + gran - 1) / gran;
    const int notify = rep & 1 ? FKV_NOTIFY_POLLING : FKV_NOTIFY_HOSTFUNC;
    const uint64_t before = launches();
    REQUIRE(g.restore(rng, pick(rng, 1, pool), gran, notify) == FKV_OK, "seed %llu", (unsigned long long)seed);
    if (batches > 1)
      REQUIRE(launches() - before == (uint64_t)g.ranks, "seed %llu: not one launch a GPU",
              (unsigned long long)seed);
    for (int l = 0; l < g.layers; ++l) {
      REQUIRE(fkv_layerwise_wait_layer(g.g, 0, l, consumer) == FKV_OK, "wait_layer");
      REQUIRE(hipMemcpyAsync(seen[l].data(), g.dev[l], g.layer_bytes(), hipMemcpyDeviceToHost, consumer) ==
                  hipSuccess, "consumer copy");
    }
    REQUIRE(hipStreamSynchronize(consumer) == hipSuccess, "consumer");
    REQUIRE(fkv_layerwise_synchronize(g.g) == FKV_OK, "synchronize");
    g.check("restore");
    for (int l = 0; l < g.layers; ++l)
      REQUIRE(seen[l] == g.model[l], "seed %llu: the consumer saw other bytes of layer %d",
              (unsigned long long)seed, l);
    for (size_t i = 0; i < g.fds.size(); ++i)
      REQUIRE(g.units(i) == 1, "seed %llu: eventfd %zu", (unsigned long long)seed, i);
    std::vector<float> ms(batches);
    int32_t count = 0;
    REQUIRE(fkv_layerwise_batch_times_ms(g.g, ms.data(), batches, &count) == FKV_OK && count == batches,
            "batch times");
    REQUIRE(std::is_sorted(ms.begin(), ms.end()), "batch times out of order");
  }
  REQUIRE(hipStreamDestroy(consumer) == hipSuccess, "stream");
  g.destroy();
}

// A restore that is held up for minutes by other work on its queue: its consumer waits, and goes
// on without the layer only when the host has found that the launch ended in an error.
void held_up_case(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, 1, 3, 1, 3, 8192);
  hipStream_t consumer = nullptr;
  REQUIRE(hipStreamCreateWithFlags(&consumer, hipStreamNonBlocking) == hipSuccess, "stream");
  std::vector<uint8_t> seen(g.layer_bytes());
  for (int rep = 0; rep < 3; ++rep) {
    const bool fails = rep == 1;
    g.refill(rng);
    fkv_emulated_hold_kernels(1);
    REQUIRE(g.restore(rng, 3, 1, FKV_NOTIFY_POLLING) == FKV_OK, "restore");
    REQUIRE(fkv_layerwise_wait_layer(g.g, 0, 2, consumer) == FKV_OK, "wait_layer");
    REQUIRE(hipMemcpyAsync(seen.data(), g.dev[2], g.layer_bytes(), hipMemcpyDeviceToHost, consumer) ==
                hipSuccess, "consumer copy");
    fkv_emulated_clock_speed(100000); // ten minutes of the device's clock in 6 ms
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    REQUIRE(hipStreamQuery(consumer) == hipErrorNotReady, "the consumer went on without its layer");
    if (fails) {
      fkv_emulated_fail(8, 0, 8);
      REQUIRE(fkv_layerwise_synchronize(g.g) != FKV_OK, "the stream's error is reported");
      fkv_emulated_fail(8, 0, 0);
      REQUIRE(hipStreamSynchronize(consumer) == hipSuccess, "nobody waits for a launch that failed");
    }
    fkv_emulated_hold_kernels(0);
    fkv_emulated_clock_speed(1);
    // (what the poller saw of the error is reported by this call)
    REQUIRE((fkv_layerwise_synchronize(g.g) == FKV_OK) == !fails, "synchronize");
    REQUIRE(hipStreamSynchronize(consumer) == hipSuccess && hipDeviceSynchronize() == hipSuccess, "end");
    g.check("held up");
    REQUIRE(fails || seen == g.model[2], "the consumer saw other bytes");
    for (size_t i = 0; i < g.fds.size(); ++i)
      (void)g.units(i);
  }
  REQUIRE(hipStreamDestroy(consumer) == hipSuccess, "stream");
  g.destroy();
}

// While some thread captures a stream the runtime does not answer whether an event has been
// reached: that is no error of the restore, and nobody is let go for it.
void no_answer_case(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, 1, 3, 1, 3, 8192);
  hipStream_t consumer = nullptr;
  REQUIRE(hipStreamCreateWithFlags(&consumer, hipStreamNonBlocking) == hipSuccess, "stream");
  std::vector<uint8_t> seen(g.layer_bytes());
  for (int notify : {FKV_NOTIFY_POLLING, FKV_NOTIFY_HOSTFUNC}) {
    g.refill(rng);
    fkv_emulated_hold_kernels(1);
    fkv_emulated_fail(9, 0, 1000000);
    std::thread call([&] { REQUIRE(g.restore(rng, 3, 1, notify) == FKV_OK, "restore"); });
    if (notify == FKV_NOTIFY_POLLING) {
      call.join();
      REQUIRE(fkv_layerwise_wait_layer(g.g, 0, 2, consumer) == FKV_OK, "wait_layer");
      REQUIRE(hipMemcpyAsync(seen.data(), g.dev[2], g.layer_bytes(), hipMemcpyDeviceToHost, consumer) ==
                  hipSuccess, "consumer copy");
    }
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    if (notify == FKV_NOTIFY_POLLING)
      REQUIRE(hipStreamQuery(consumer) == hipErrorNotReady, "the consumer went on without its layer");
    fkv_emulated_hold_kernels(0);
    if (notify == FKV_NOTIFY_HOSTFUNC)
      call.join();
    REQUIRE(fkv_layerwise_synchronize(g.g) == FKV_OK, "synchronize");
    fkv_emulated_fail(9, 0, 0);
    REQUIRE(hipStreamSynchronize(consumer) == hipSuccess, "consumer");
    g.check("no answer");
    REQUIRE(notify == FKV_NOTIFY_HOSTFUNC || seen == g.model[2], "the consumer saw other bytes");
    for (size_t i = 0; i < g.fds.size(); ++i)
      REQUIRE(g.units(i) == 1, "eventfd %zu", i);
  }
  REQUIRE(hipStreamDestroy(consumer) == hipSuccess, "stream");
  g.destroy();
}

// A call that returns when everything has landed (HOSTFUNC) leaves nothing running: the times of
// its batches are there, and whatever it used is free.
void drained_case(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, 2, 3, 1, 3, 8192);
  fkv_emulated_kernel_tail(3000);
  for (int rep = 0; rep < 3; ++rep) {
    g.refill(rng);
    REQUIRE(g.restore(rng, 2, 1, FKV_NOTIFY_HOSTFUNC) == FKV_OK, "restore");
    float ms[3];
    int32_t count = 0;
    REQUIRE(fkv_layerwise_batch_times_ms(g.g, ms, 3, &count) == FKV_OK && count == 3,
            "the call returned before its streams had drained");
    g.check("drained");
  }
  fkv_emulated_kernel_tail(0);
  g.destroy();
}

// kernel_alt_stream_kb chosen by the caller: batch by batch, on one stream (0) or two.
void by_policy(uint64_t seed) {
  Rng rng(seed);
  for (int layers : {3, 13}) // fewer and more batches than two streams are worth
    for (int alt_kb : {-1, 0, 1, 4096}) {
      Group g(rng, 1, layers, 1, 2, 8192);
      set_policy(alt_kb);
      const uint64_t before = launches();
      REQUIRE(g.restore(rng, 2, 1, FKV_NOTIFY_HOSTFUNC) == FKV_OK, "restore");
      REQUIRE(launches() - before == (uint64_t)(alt_kb < 0 ? 1 : layers),
              "kernel_alt_stream_kb %d, %d batches: %d launches", alt_kb, layers, (int)(launches() - before));
      g.check("by policy");
      g.destroy();
    }
  set_policy();
}

// Next to a transfer from the GPU a restore asks for no more workgroups than a launch per batch
// does: the writer pays for them.  (Workgroups launched, confined ones of which half the XCDs'
// stay; only where the kernel itself runs.)
void next_to_a_put(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, 1, 8, 1, 16, 8192);
  std::vector<uint64_t> ptrs;
  for (uint8_t *d : g.dev)
    ptrs.push_back((uint64_t)(uintptr_t)d);
  std::vector<int64_t> ids{0};
  hipStream_t other = nullptr;
  REQUIRE(hipStreamCreateWithFlags(&other, hipStreamNonBlocking) == hipSuccess, "stream");
  fkv_launch_policy p{};
  REQUIRE(fkv_launch_policy_get(0, &p) == FKV_OK, "policy");
  p.busy_window_ms = 20000; // a put counts for as long as this program runs
  REQUIRE(fkv_launch_policy_set(0, &p) == FKV_OK, "policy");
  uint8_t *sink = nullptr;
  REQUIRE(hipHostMalloc((void **)&sink, (size_t)g.block(), 0) == hipSuccess, "sink");
  fkv_transfer_desc d{};
  d.backend = FKV_BACKEND_VLLM;
  d.num_layers_total = d.num_layers = d.num_gpu_tensor_ptrs = g.layers;
  d.gpu_tensor_ptrs = ptrs.data();
  d.device = 0;
  d.gpu_kv_stride = d.gpu_layer_stride = (int64_t)g.layer_bytes();
  d.gpu_block_stride = d.cpu_kv_stride = d.cpu_layer_stride = d.chunk_size = g.chunk;
  d.cpu_ptr = sink;
  d.cpu_block_stride = g.block();
  d.kv_dim = d.num_blocks = d.sync = 1;
  d.gpu_block_ids = d.cpu_block_ids = ids.data();
  d.transfer_num_cta = 4;
  fkv_ce_config_default(&d.ce);
  REQUIRE(fkv_transfer_kv_blocks(&d, other) == FKV_OK, "put");
  auto workgroups = [&](int alt_kb) {
    p.kernel_alt_stream_kb = alt_kb;
    REQUIRE(fkv_launch_policy_set(0, &p) == FKV_OK, "policy");
    const unsigned long long before = fkv_emulated_workgroups_run();
    const uint64_t launched = launches();
    g.refill(rng);
    REQUIRE(g.restore(rng, 16, 4, FKV_NOTIFY_HOSTFUNC) == FKV_OK, "restore");
    g.check("next to a put");
    return (fkv_emulated_workgroups_run() - before) / (launches() - launched);
  };
  const unsigned long long batches = workgroups(0), single = workgroups(-1);
  REQUIRE(single <= batches, "%llu workgroups, %llu of a launch per batch", single, batches);
  REQUIRE(hipHostFree(sink) == hipSuccess && hipStreamDestroy(other) == hipSuccess, "free");
  set_policy();
  g.destroy();
}

// The words of a launch may reach the host a little after the event behind it is seen: no error.
void late_words_case(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, 1, 3, 1, 3, 8192);
  fkv_emulated_late_words(1000);
  for (int rep = 0; rep < 6; ++rep) {
    g.refill(rng);
    REQUIRE(g.restore(rng, 3, 1, rep & 1 ? FKV_NOTIFY_POLLING : FKV_NOTIFY_HOSTFUNC) == FKV_OK, "restore");
    REQUIRE(fkv_layerwise_synchronize(g.g) == FKV_OK, "synchronize");
    g.check("late words");
    for (size_t i = 0; i < g.fds.size(); ++i)
      REQUIRE(g.units(i) == 1, "rep %d: eventfd %zu", rep, i);
  }
  fkv_emulated_late_words(0);
  g.destroy();
}

// Groups that restore at the same time, each from a thread of its own.
void several_at_once(uint64_t seed) {
  std::vector<std::thread> threads;
  for (int t = 0; t < 3; ++t)
    threads.emplace_back([seed, t] {
      Rng rng(seed * 8 + t);
      for (int k = 0; k < 2; ++k) { // the second group takes words that another one gave back
        Group g(rng, 1, pick(rng, 2, 6), 1, 4, 8192);
        for (int rep = 0; rep < 3; ++rep) {
          g.refill(rng);
          REQUIRE(g.restore(rng, pick(rng, 1, 4), 1, rep & 1) == FKV_OK, "restore");
          REQUIRE(fkv_layerwise_synchronize(g.g) == FKV_OK, "synchronize");
          g.check("several at once");
        }
        g.destroy();
      }
    });
  for (auto &t : threads)
    t.join();
}

// The runtime refuses something part-way: the restore fails or makes up for it, and the next
// one is whole.
void refused_case(uint64_t seed) {
  Rng rng(seed);
  Group g(rng, pick(rng, 1, 2), pick(rng, 2, 5), 1, 4, 8192);
  for (int rep = 0; rep < 4; ++rep) {
    const bool inject = rep % 2 == 0;
    g.refill(rng);
    if (inject)
      fkv_emulated_fail(pick(rng, 0, 7), pick(rng, 0, 5), pick(rng, 1, 3));
    const int rc = g.restore(rng, pick(rng, 1, 4), 1, pick(rng, 0, 1));
    const int src = fkv_layerwise_synchronize(g.g);
    for (int c = 0; c < 8; ++c)
      fkv_emulated_fail(c, 0, 0);
    const bool whole = rc == FKV_OK && src == FKV_OK;
    REQUIRE(whole || inject, "seed %llu rep %d: a clean restore failed", (unsigned long long)seed, rep);
    if (whole)
      g.check("refused calls");
    for (size_t i = 0; i < g.fds.size(); ++i) {
      const int units = g.units(i);
      REQUIRE(whole ? units == 1 : units <= 1, "seed %llu: eventfd %zu has %d", (unsigned long long)seed, i, units);
    }
    for (size_t i = 0; i < g.dev.size(); ++i)
      memcpy(g.model[i].data(), g.dev[i], g.layer_bytes());
  }
  g.destroy();
}

} // namespace

int main(int argc, char **argv) {
  const int cases = argc > 1 ? atoi(argv[1]) : 20;
  set_policy();
  first_words(20400);
  for (int i = 0; i < cases; ++i)
    seeded_case(21000 + i);
  held_up_case(20500);
  no_answer_case(20550);
  late_words_case(20580);
  drained_case(20600);
  by_policy(20700);
  next_to_a_put(20800);
  for (int i = 0; i < (cases + 3) / 4; ++i)
    several_at_once(22000 + i);
  for (int i = 0; i < cases; ++i)
    refused_case(23000 + i);
  printf("ok: %d groups of single-launch restores, kernels from their sources: %s\n", cases,
         fkv_emulated_workgroups_run() ? "yes" : "no");
  return 0;
}
