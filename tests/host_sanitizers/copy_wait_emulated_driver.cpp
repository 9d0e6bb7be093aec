// Waiting transfers of several threads that start together, the kernels from their sources on the CPU
// device model: the words they wait for are allocated once, not once a thread, and none of them waits for
// another one's stream.
#include <hip/hip_runtime.h>

#include "fkv_transfer.h"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#define REQUIRE(cond, ...)                                                                          \
  do {                                                                                              \
    if (!(cond)) {                                                                                  \
      fprintf(stderr, "copy_wait_emulated_driver: " __VA_ARGS__);                                   \
      fprintf(stderr, " [%s:%d]\n", __FILE__, __LINE__);                                            \
      _Exit(1);                                                                                     \
    }                                                                                               \
  } while (0)

extern "C" long fkv_emulated_small_pinned_allocations();
extern "C" void fkv_emulated_hold_kernels(int on);

namespace {

constexpr int kThreads = 12, kChunk = 64;

struct Caller {
  hipStream_t stream = nullptr;
  uint8_t *gpu = nullptr, *host = nullptr;
  uint64_t table[1];
  int64_t id[1] = {0};
  fkv_transfer_desc d{};
  void make(int t) {
    REQUIRE(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) == hipSuccess, "stream");
    REQUIRE(hipMalloc((void **)&gpu, kChunk) == hipSuccess, "device memory");
    REQUIRE(hipHostMalloc((void **)&host, kChunk, 0) == hipSuccess, "host memory");
    table[0] = (uint64_t)(uintptr_t)gpu;
    d.backend = FKV_BACKEND_VLLM;
    d.num_layers_total = 1, d.gpu_tensor_ptrs = table, d.num_gpu_tensor_ptrs = 1, d.device = -1;
    d.gpu_kv_stride = d.gpu_block_stride = d.gpu_layer_stride = kChunk;
    d.cpu_ptr = host, d.cpu_kv_stride = d.cpu_layer_stride = d.cpu_block_stride = kChunk;
    d.chunk_size = kChunk, d.num_layers = 1, d.kv_dim = 1, d.num_blocks = 1;
    d.gpu_block_ids = d.cpu_block_ids = id;
    d.is_host_to_device = t & 1;
    fkv_ce_config_default(&d.ce);
  }
  void call(int sync, int value) {
    memset(d.is_host_to_device ? host : gpu, value, kChunk);
    d.sync = sync;
    REQUIRE(fkv_transfer_kv_blocks(&d, stream) == FKV_OK, "%s", fkv_last_error());
  }
  void check(int value) {
    const uint8_t *there = d.is_host_to_device ? gpu : host;
    for (int i = 0; i < kChunk; ++i)
      REQUIRE(there[i] == value, "byte %d: %d, not %d", i, there[i], value);
  }
};

// All of them wait for a device that does not get to it for a while.  Returns the allocations meanwhile.
long together(std::vector<Caller> &callers, int value) {
  const long before = fkv_emulated_small_pinned_allocations();
  fkv_emulated_hold_kernels(1);
  std::atomic<int> running{0}, over{0};
  std::vector<std::thread> threads;
  for (Caller &c : callers)
    threads.emplace_back([&, value] {
      running.fetch_add(1);
      c.call(1, value);
      c.check(value);
      over.fetch_add(1);
    });
  while (running.load() < (int)callers.size())
    std::this_thread::yield();
  std::this_thread::sleep_for(std::chrono::milliseconds(300));
  REQUIRE(over.load() == 0, "a call returned before its kernel ran");
  fkv_emulated_hold_kernels(0);
  for (auto &t : threads)
    t.join();
  return fkv_emulated_small_pinned_allocations() - before;
}

} // namespace

int main() {
  std::vector<Caller> callers(kThreads);
  for (int t = 0; t < kThreads; ++t)
    callers[t].make(t);
  callers[0].call(0, 3); // what the library measures and sets up on first use, without a wait for a word
  REQUIRE(hipStreamSynchronize(callers[0].stream) == hipSuccess, "stream");
  callers[0].check(3);
  const long cold = together(callers, 7);
  REQUIRE(cold == 1, "%ld allocations for %d calls that start together", cold, kThreads);
  for (int round = 8; round < 12; ++round) {
    const long warm = together(callers, round);
    REQUIRE(warm == 0, "%ld allocations for calls that find words", warm);
  }
  for (Caller &c : callers)
    REQUIRE(hipStreamDestroy(c.stream) == hipSuccess && hipFree(c.gpu) == hipSuccess &&
                hipHostFree(c.host) == hipSuccess, "given back");
  printf("ok: %d threads waiting at once\n", kThreads);
  return 0;
}
