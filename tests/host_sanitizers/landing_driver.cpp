// The counting and announcing of batches by the wavefronts of a single-launch restore
// (fkv_landing.h), without the copies: wavefronts as state machines that take turns in a seeded
// order, some of them slow, every word checked after every step.
#include "cpu_device_model.h"

#include "fkv_landing.h"

#include <cstdio>
#include <cstdlib>
#include <random>
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

struct Words {
  std::vector<uint32_t> arrived;
  std::vector<uint64_t> landed, landed_host, ticks;
  fkv::LayersLaunch t{};
  Words(int batches, int ranges) : arrived(batches), landed(batches), landed_host(batches), ticks(batches) {
    t.batches = batches, t.ranges = ranges;
    t.arrived = arrived.data(), t.landed = landed.data();
    t.landed_host = landed_host.data(), t.tick_host = ticks.data();
  }
  int parts() const { return t.ranges * t.batches; }
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
  Words w(pick(rng, 1, 12), pick(rng, 1, 5));
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
      bool whole = true; // every batch so far has all its ranges counted
      for (int b = 0; b < w.t.batches; ++b) {
        whole = whole && counted[b] == w.t.ranges;
        REQUIRE(whole || (w.landed[b] < w.t.epoch && w.landed_host[b] < w.t.epoch),
                "seed %llu: batch %d of %d announced before all up to it had landed",
                (unsigned long long)seed, b, w.t.batches);
      }
      busy = false;
      for (const Wavefront &v : wave)
        busy = busy || v.at != Wavefront::kDone;
    }
    for (int b = 0; b < w.t.batches; ++b)
      REQUIRE(w.landed[b] == w.t.epoch && w.landed_host[b] == w.t.epoch && w.arrived[b] == 0 &&
                  (b == 0 || w.ticks[b] >= w.ticks[b - 1]),
              "seed %llu: batch %d at the end", (unsigned long long)seed, b);
  }
}

} // namespace

int main(int argc, char **argv) {
  const int cases = argc > 1 ? atoi(argv[1]) : 100;
  for (int i = 0; i < cases; ++i)
    turns(31000 + i);
  printf("ok: %d landings by turns\n", cases);
  return 0;
}
