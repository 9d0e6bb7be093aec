// The counting and announcing of batches by the wavefronts of a single-launch restore
// (fkv_landing.h) and the streams that wait for them, without the copies: wavefronts as state machines that take turns in a seeded
// order, some of them slow, every word checked after every step; and as host threads, for ThreadSanitizer.
#include "cpu_device_model.h"

#include "fkv_landing.h"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#define REQUIRE(cond, ...)                                                                          \
  do {                                                                                              \
    if (!(cond)) {                                                                                  \
      fprintf(stderr, "landing_driver: " __VA_ARGS__);                                              \
      fprintf(stderr, " [%s:%d]\n", __FILE__, __LINE__);                                            \
      exit(1);                                                                                      \
    }                                                                                               \
  } while (0)

namespace {

using Rng = std::mt19937_64;
int pick(Rng &rng, int lo, int hi) { return lo + (int)(rng() % (uint64_t)(hi - lo + 1)); }

// How a restore is cut: no empty range, whatever the last batch is; no range of more than 16 or so
// slices, and enough of them for every wavefront, as far as there are slices.
void cuts(uint64_t seed) {
  Rng rng(seed);
  const int64_t pairs = pick(rng, 1, 64), batches = pick(rng, 1, 40), last = pick(rng, 1, (int)pairs),
                per_pair = std::vector<int>{1, 2, 7, 100, 5000}[pick(rng, 0, 4)], working = pick(rng, 1, 96);
  const fkv::LayersCut c = fkv::cut_layers(batches, pairs, last, per_pair, working);
  const int64_t slices = pairs * per_pair;
  REQUIRE(c.ranges >= 1 && c.ranges <= slices && c.last_ranges >= 1 && c.last_ranges <= last * per_pair &&
              c.last_ranges <= c.ranges, "seed %llu: an empty range", (unsigned long long)seed);
  REQUIRE(c.ranges == slices || (c.ranges * 32 > slices && c.ranges * batches >= 2 * working),
          "seed %llu: %lld ranges of %lld slices for %lld wavefronts", (unsigned long long)seed,
          (long long)c.ranges, (long long)slices, (long long)working);
  REQUIRE(c.last_ranges == last * per_pair || c.last_ranges * pairs >= c.ranges * last,
          "seed %llu: longer ranges in the last batch", (unsigned long long)seed);
}

struct Words {
  std::vector<uint32_t> arrived;
  std::vector<uint64_t> landed, landed_host, ticks;
  fkv::LayersLaunch t{};
  Words(int batches, int ranges, int last_ranges) : arrived(batches), landed(batches), landed_host(batches), ticks(batches) {
    t.batches = batches, t.ranges = ranges, t.last_ranges = last_ranges;
    t.arrived = arrived.data(), t.landed = landed.data();
    t.landed_host = landed_host.data(), t.tick_host = ticks.data();
  }
  int parts() const { return t.ranges * (t.batches - 1) + t.last_ranges; }
  int batch_of(int part) const { return part / t.ranges; }
};

// What the kernel does with a range, in the steps between which others get their turn.
struct Wavefront {
  fkv::Landing landing;
  enum { kClaim, kArrived, kStored, kLast, kDone } at = kClaim;
  int part = -1;
  explicit Wavefront(const Words &w) : landing(w.t, true) {}
  void step(const Words &w, int *next, std::vector<int> *counted) {
    auto count = [&] {
      ++(*counted)[landing.copied];
      landing.count();
    };
    switch (at) {
    case kClaim:
      part = (*next)++;
      at = part < w.parts() ? kArrived : kLast;
      break;
    case kArrived: // the first vectors of this range are here: so are the stores of the one before
      landing.announce();
      if (landing.copied >= 0)
        count();
      at = kStored;
      break;
    case kStored:
      landing.announce();
      landing.copied = w.batch_of(part);
      at = kClaim;
      break;
    case kLast:
      landing.announce();
      if (landing.copied >= 0) {
        count();
        break;
      }
      at = kDone;
      break;
    case kDone:
      break;
    }
  }
};

void turns(uint64_t seed) {
  Rng rng(seed);
  const int ranges = pick(rng, 1, 5);
  Words w(pick(rng, 1, 12), ranges, pick(rng, 1, ranges));
  const int waves = pick(rng, 1, 9);
  for (w.t.epoch = 1; w.t.epoch <= 3; ++w.t.epoch) {
    std::vector<Wavefront> wave(waves, Wavefront(w));
    std::vector<int> counted(w.t.batches, 0), speed(waves);
    for (int &s : speed)
      s = pick(rng, 0, 3) ? 100 : 3; // of a hundred turns
    int next = 0;
    for (bool busy = true; busy;) {
      const int i = pick(rng, 0, waves - 1);
      if (pick(rng, 1, 100) <= speed[i])
        wave[i].step(w, &next, &counted);
      for (int b = 0; b < w.t.batches; ++b)
        REQUIRE(counted[b] == (int)w.t.ranges_of(b) || (w.landed[b] < w.t.epoch && w.landed_host[b] < w.t.epoch),
                "seed %llu: batch %d of %d announced before it had landed",
                (unsigned long long)seed, b, w.t.batches);
      busy = false;
      for (const Wavefront &v : wave)
        busy = busy || v.at != Wavefront::kDone;
    }
    for (int b = 0; b < w.t.batches; ++b)
      REQUIRE(w.landed[b] == w.t.epoch && w.landed_host[b] == w.t.epoch && w.arrived[b] == 0,
              "seed %llu: batch %d at the end", (unsigned long long)seed, b);
  }
}

// Wavefronts as host threads, copies as plain stores: whoever has seen the words of a batch and of
// all before it reads every byte of them.
void threads(uint64_t seed) {
  Rng rng(seed);
  const int ranges = pick(rng, 1, 6);
  Words w(pick(rng, 1, 10), ranges, pick(rng, 1, ranges));
  w.t.epoch = 7;
  std::vector<int> bytes(w.parts(), 0); // what the copies write: plain memory
  std::atomic<int> next{0}, ready{0};
  std::vector<std::thread> all;
  for (int i = 0; i < 6; ++i)
    all.emplace_back([&] {
      fkv::Landing landing(w.t, true);
      ready.fetch_add(1, std::memory_order_relaxed);
      while (ready.load(std::memory_order_relaxed) < 6) // all of them get some of the work
        std::this_thread::yield();
      for (int part; (part = next.fetch_add(1, std::memory_order_relaxed)) < w.parts();) {
        landing.announce();
        if (landing.copied >= 0)
          landing.count();
        bytes[part] = part + 1;
        landing.announce();
        landing.copied = w.batch_of(part);
        std::this_thread::yield();
      }
      landing.announce();
      if (landing.copied >= 0)
        landing.count();
      landing.announce();
    });
  for (int reader = 0; reader < 2; ++reader)
    all.emplace_back([&, only = pick(rng, 0, w.t.batches - 1), host = reader == 1] {
      for (int b = 0; b <= only; ++b)
        while (__atomic_load_n((host ? w.t.landed_host : w.t.landed) + b, __ATOMIC_ACQUIRE) < w.t.epoch)
          std::this_thread::yield();
      for (int part = 0; part < w.parts() && w.batch_of(part) <= only; ++part)
        REQUIRE(bytes[part] == part + 1, "seed %llu: batch %d, part %d", (unsigned long long)seed, only, part);
    });
  for (auto &t : all)
    t.join();
}

// Words written in any order: a stream that waits for one batch goes on when every word up to
// that one is there, at the device's words and at those the host sees.
void any_order(uint64_t seed, hipStream_t stream) {
  Rng rng(seed);
  Words w(pick(rng, 1, 150), 1, 1);
  w.t.epoch = 5;
  uint64_t given_up = 4;
  hipEvent_t behind = nullptr;
  REQUIRE(hipEventCreate(&behind) == hipSuccess, "event");
  std::vector<int> order(w.t.batches);
  for (int b = 0; b < w.t.batches; ++b)
    order[b] = b;
  std::shuffle(order.begin(), order.end(), rng);
  const int only = pick(rng, 0, w.t.batches - 1), begun = pick(rng, 0, w.t.batches);
  auto write = [&](int k) {
    __atomic_store_n(&w.landed[order[k]], w.t.epoch, __ATOMIC_RELEASE);
    __atomic_store_n(&w.landed_host[order[k]], w.t.epoch, __ATOMIC_RELEASE);
  };
  for (int k = 0; k < begun; ++k)
    write(k);
  REQUIRE(fkv::layers_device->wait(w.t.landed, w.t.landed_host, only + 1, w.t.epoch, &given_up, 0, behind,
                                   stream) == FKV_OK, "wait");
  for (int k = begun; k <= w.t.batches; ++k) {
    bool there = true;
    for (int b = 0; b <= only; ++b)
      there = there && w.landed[b] == w.t.epoch;
    if (there) {
      REQUIRE(hipStreamSynchronize(stream) == hipSuccess, "stream");
      break;
    }
    if (k % 16 == begun % 16)
      std::this_thread::sleep_for(std::chrono::milliseconds(2));
    REQUIRE(hipStreamQuery(stream) == hipErrorNotReady,
            "seed %llu: the stream went on without a batch before %d", (unsigned long long)seed, only);
    write(k);
  }
  REQUIRE(hipEventDestroy(behind) == hipSuccess, "event");
}

} // namespace

int main(int argc, char **argv) {
  const int cases = argc > 1 ? atoi(argv[1]) : 100;
  for (int i = 0; i < 20 * cases; ++i)
    cuts(30000 + i);
  for (int i = 0; i < cases; ++i)
    turns(31000 + i);
  for (int i = 0; i < cases; ++i)
    threads(32000 + i);
  hipStream_t stream = nullptr;
  REQUIRE(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) == hipSuccess, "stream");
  for (int i = 0; i < cases / 4; ++i)
    any_order(33000 + i, stream);
  REQUIRE(hipStreamDestroy(stream) == hipSuccess, "stream");
  printf("ok: %d landings by turns and by threads\n", cases);
  return 0;
}
