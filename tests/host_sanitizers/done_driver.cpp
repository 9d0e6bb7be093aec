// The counts by which a launch tells whoever waits for it that everything has been copied
// (fkv_done.h), without the copies: workgroups as state machines that take turns in a seeded order, on several XCDs,
// some of them dispatched late, some of them long in their release, launch after launch on one set
// of counts while workgroups of the launches before are still around; and as host threads, for ThreadSanitizer.
#include "cpu_device_model.h"

#include "fkv_done.h"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#define REQUIRE(cond, ...)                                                                          \
  do {                                                                                              \
    if (!(cond)) {                                                                                  \
      fprintf(stderr, "done_driver: " __VA_ARGS__);                                                 \
      fprintf(stderr, " [%s:%d]\n", __FILE__, __LINE__);                                            \
      exit(1);                                                                                      \
    }                                                                                               \
  } while (0)

namespace {

using Rng = std::mt19937_64;
int pick(Rng &rng, int lo, int hi) { return lo + (int)(rng() % (uint64_t)(hi - lo + 1)); }

// Nobody at work, everything reported.
bool at_rest(const fkv::DoneCounts &c) {
  for (int x = 0; x < 16; ++x)
    if (c.of_xcd[x] != c.reported[x] * fkv::kDoneShare)
      return false;
  return c.all == 0;
}

enum ShareState { kNotThere, kInL2, kReleased };
struct Launch {
  fkv::CopyDone done;
  bool to_host = true, claimed = true;
  int workgroups = 0, next = 0;
  std::vector<ShareState> shares;
  std::vector<int> xcd_of; // of a share: whose L2 holds it
};

// What the kernel does, in the steps between which others get their turn.
struct Workgroup {
  enum { kNotDispatched, kClaim, kBegin, kCopy, kLeave, kRelease, kTake, kReport, kOver } at = kNotDispatched;
  Launch *l;
  int index, xcd, late, release_turns, part = -1;
  uint32_t copied = 0, to_report = 0;
  uint64_t far = 0;
  std::vector<int> releasing; // shares in the L2 when the release began

  void step() {
    switch (at) {
    case kNotDispatched:
      if (--late < 0)
        at = kClaim;
      break;
    case kClaim:
      if (l->claimed)
        part = l->next++;
      else
        part = copied == 0 ? index : (int)l->shares.size();
      at = part < (int)l->shares.size() ? (copied == 0 && l->to_host ? kBegin : kCopy)
                                        : (copied ? kLeave : kOver);
      break;
    case kBegin:
      fkv::begin_on_xcd(l->done, (uint32_t)xcd);
      at = kCopy;
      break;
    case kCopy:
      l->shares[part] = kInL2;
      l->xcd_of[part] = l->to_host ? xcd : index; // into HBM every workgroup releases its own
      ++copied;
      at = kClaim;
      break;
    case kLeave:
      far = l->to_host ? fkv::leave_xcd(l->done, (uint32_t)xcd, copied) : copied;
      if (far)
        for (int s = 0; s < (int)l->shares.size(); ++s)
          if (l->shares[s] == kInL2 && l->xcd_of[s] == (l->to_host ? xcd : index))
            releasing.push_back(s);
      at = far ? kRelease : kOver;
      break;
    case kRelease:
      if (--release_turns > 0)
        break;
      for (int s : releasing)
        l->shares[s] = kReleased;
      at = kTake;
      break;
    case kTake:
      to_report = l->to_host ? fkv::newly_released(l->done, (uint32_t)xcd, far) : copied;
      at = kReport;
      break;
    case kReport:
      fkv::report_copied(l->done, to_report, (uint32_t)l->shares.size());
      at = kOver;
      break;
    case kOver:
      break;
    }
  }
};

void turns(uint64_t seed) {
  Rng rng(seed);
  fkv::DoneCounts counts{};
  uint64_t word = 0;
  const int launches = pick(rng, 2, 5), xcds = pick(rng, 1, 3);
  std::vector<Launch> made(launches); // workgroups point into it
  std::vector<Workgroup> all;
  for (int n = 0; n < launches; ++n) {
    Launch &l = made[n];
    l.done.count = &counts, l.done.word = &word, l.done.epoch = (uint64_t)n + 1;
    l.to_host = pick(rng, 0, 7) != 0;
    l.claimed = pick(rng, 0, 3) != 0;
    l.workgroups = pick(rng, 1, 8);
    const int shares = l.claimed ? pick(rng, 1, 14) : l.workgroups;
    l.shares.assign(shares, kNotThere);
    l.xcd_of.assign(shares, -1);
    for (int i = 0; i < l.workgroups; ++i) {
      Workgroup w;
      w.l = &l, w.index = i, w.xcd = pick(rng, 0, xcds - 1);
      w.late = pick(rng, 0, 2) ? 0 : pick(rng, 1, 60);
      w.release_turns = pick(rng, 0, 2) ? pick(rng, 1, 3) : pick(rng, 4, 80);
      all.push_back(w);
    }
    long left = 200000;
    while (word < l.done.epoch) { // whoever waits; the workgroups of earlier launches may go on
      REQUIRE(--left > 0, "seed %llu: launch %d of %d never says that it is over", (unsigned long long)seed, n, launches);
      all[(size_t)(rng() % all.size())].step();
      REQUIRE(word <= l.done.epoch, "seed %llu: word %llu", (unsigned long long)seed, (unsigned long long)word);
    }
    for (int s = 0; s < shares; ++s)
      REQUIRE(l.shares[s] == kReleased, "seed %llu: launch %d of %d said to be over without share %d of %d",
              (unsigned long long)seed, n, launches, s, shares);
    REQUIRE(at_rest(counts), "seed %llu: counts behind launch %d", (unsigned long long)seed, n);
    for (int k = pick(rng, 0, 30); k > 0; --k)
      all[(size_t)(rng() % all.size())].step();
  }
  for (bool busy = true; busy;) {
    busy = false;
    for (Workgroup &w : all) {
      w.step();
      busy = busy || w.at != Workgroup::kOver;
    }
  }
  REQUIRE(at_rest(counts) && word == (uint64_t)launches, "seed %llu: at the end", (unsigned long long)seed);
}

// Workgroups as host threads, copies as plain stores: whoever has seen the word reads every byte.
void threads(uint64_t seed) {
  Rng rng(seed);
  constexpr int kWorkgroups = 6, kLaunches = 5;
  fkv::DoneCounts counts{};
  uint64_t word = 0;
  struct One {
    std::vector<int> bytes; // what the copies write: plain memory
    std::atomic<int> next{0};
    bool to_host = true;
  } made[kLaunches];
  for (One &l : made) {
    l.bytes.assign(pick(rng, 1, 30), 0);
    l.to_host = pick(rng, 0, 3) != 0;
  }
  std::atomic<int> launched{0};
  std::vector<std::thread> all;
  for (int i = 0; i < kWorkgroups; ++i)
    all.emplace_back([&, xcd = (uint32_t)pick(rng, 0, 1)] {
      for (int n = 0; n < kLaunches; ++n) {
        One &l = made[n];
        while (launched.load(std::memory_order_acquire) <= n)
          std::this_thread::yield();
        fkv::CopyDone done;
        done.count = &counts, done.word = &word, done.epoch = (uint64_t)n + 1;
        uint32_t copied = 0;
        for (int part; (part = l.next.fetch_add(1, std::memory_order_relaxed)) < (int)l.bytes.size();) {
          if (copied == 0 && l.to_host)
            fkv::begin_on_xcd(done, xcd);
          l.bytes[part] = part + 1;
          ++copied;
          std::this_thread::yield();
        }
        if (copied == 0)
          continue;
        const uint64_t far = l.to_host ? fkv::leave_xcd(done, xcd, copied) : copied;
        if (far == 0)
          continue;
        std::this_thread::yield();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
        std::this_thread::yield();
        fkv::report_copied(done, l.to_host ? fkv::newly_released(done, xcd, far) : copied,
                           (uint32_t)l.bytes.size());
      }
    });
  for (int n = 0; n < kLaunches; ++n) {
    launched.store(n + 1, std::memory_order_release);
    uint64_t at;
    while ((at = __atomic_load_n(&word, __ATOMIC_ACQUIRE)) < (uint64_t)n + 1)
      std::this_thread::yield();
    REQUIRE(at == (uint64_t)n + 1, "seed %llu: word", (unsigned long long)seed);
    for (int part = 0; part < (int)made[n].bytes.size(); ++part)
      REQUIRE(made[n].bytes[part] == part + 1, "seed %llu: launch %d, share %d", (unsigned long long)seed, n, part);
  }
  for (auto &t : all)
    t.join();
  REQUIRE(at_rest(counts) && word == kLaunches, "seed %llu: at the end", (unsigned long long)seed);
}

} // namespace

int main(int argc, char **argv) {
  const int cases = argc > 1 ? atoi(argv[1]) : 1000;
  for (int i = 0; i < 10 * cases; ++i)
    turns(41000 + i);
  for (int i = 0; i < cases / 4; ++i)
    threads(42000 + i);
  printf("ok: %d sets of counted launches\n", cases);
  return 0;
}
