// The bookkeeping of csrc/block_cache.h against a simulated set of devices
// (CPU only).  Built and run by tests/test_block_cache.py; prints "ALL OK" and
// exits 0 on success.
#include "block_cache.h"

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#define REQUIRE(c)                                                      \
  do {                                                                  \
    if (!(c)) {                                                         \
      std::fprintf(stderr, "FAILED %s at line %d\n", #c, __LINE__);     \
      std::exit(1);                                                     \
    }                                                                   \
  } while (0)

namespace {

// Addresses are handed out by counting and freed ones are not used again
struct devices {
  struct block {
    int device;
    size_t size;
    bool busy; // work of the device may still use it
  };
  static inline std::mutex mutex;
  static inline std::map<void *, block> live;
  static inline size_t bytes = 0, limit = ~size_t(0), next = 4096;
  static inline bool refuse = false, free_fails = false; // a stream capture; a device in error
  static inline thread_local int now = 0; // a new thread's device is 0

  static bool alloc(void **p, size_t n)
  {
    std::lock_guard<std::mutex> lock(mutex);
    if (refuse || bytes + n > limit) return false;
    if (n == 0) {
      *p = nullptr;
      return true;
    }
    *p = reinterpret_cast<void *>(next);
    next += n + 4096;
    bytes += n;
    live[*p] = {now, n, false};
    return true;
  }
  static bool release(void *p)
  {
    std::lock_guard<std::mutex> lock(mutex);
    REQUIRE(live.count(p));
    bytes -= live[p].size;
    live.erase(p);
    if (free_fails) return false;
    for (auto &b : live)
      if (b.second.device == now) b.second.busy = false;
    return true;
  }
  static int current() { return now; }
};

using cache_t = mfp::block_cache<devices>;

// a block as an object of the current device gets it
void *take(cache_t &c, size_t n)
{
  void *p = c.get(n);
  REQUIRE(p);
  std::lock_guard<std::mutex> lock(devices::mutex);
  REQUIRE(devices::live.count(p));
  auto &b = devices::live[p];
  REQUIRE(b.device == devices::now); // another device's memory is not this one's
  REQUIRE(b.size >= n);
  REQUIRE(!b.busy); // nothing runs on it any more
  b.busy = true;
  return p;
}

// gives it back as an object does that waited for nothing itself
bool put(cache_t &c, void *p) { return c.put(p, false); }

constexpr size_t MB = 1u << 20;

void reuse()
{
  cache_t c;
  void *hold = take(c, 1000); // keeps the cache from emptying
  void *p = take(c, 20 * MB);
  put(c, p);
  REQUIRE(c.kept_bytes(0) >= 20 * MB && c.kept_bytes(1) == 0);
  REQUIRE(take(c, 19 * MB) == p);
  REQUIRE(c.kept_bytes(0) == 0);
  put(c, p);
  void *q = take(c, 5 * MB); // a far smaller one does not take it
  REQUIRE(q != p);
  c.trim();
  REQUIRE(c.kept_bytes(0) == 0 && devices::live.size() == 2);
  put(c, q);
  put(c, hold);
  REQUIRE(devices::live.empty()); // the last block gives everything back
}

// Where allocations are refused, kept blocks are too, and a block that is freed
// meanwhile is not kept
void refused()
{
  cache_t c;
  void *hold = take(c, 1000), *p = take(c, 20 * MB), *q = take(c, 30 * MB);
  put(c, p);
  devices::refuse = true;
  REQUIRE(!c.get(20 * MB));
  put(c, q);
  REQUIRE(!devices::live.count(q));
  devices::refuse = false;
  REQUIRE(c.kept_bytes(0) == 0);
  void *r = take(c, 20 * MB);
  put(c, r);
  devices::refuse = true;
  REQUIRE(!c.get(20 * MB) && !devices::live.count(r)); // the kept one is given back meanwhile
  devices::refuse = false;
  put(c, hold);
  REQUIRE(devices::live.empty());
}

// An object's arrays: the first is waited for, which tells that the others are
// idle too
void together()
{
  cache_t c;
  void *hold = take(c, 1000);
  void *p = take(c, 20 * MB), *q = take(c, 30 * MB);
  REQUIRE(put(c, p)); // waited
  const size_t next = devices::next;
  REQUIRE(c.put(q, true) && devices::next == next); // no token, no wait
  REQUIRE(take(c, 30 * MB) == q && take(c, 20 * MB) == p);
  // what is not known stays unknown: another device's block, a small one, a refused wait
  devices::now = 1;
  REQUIRE(!put(c, p) && !devices::live.count(p));
  devices::now = 0;
  void *small = take(c, 1000);
  REQUIRE(!put(c, small));
  devices::refuse = true;
  REQUIRE(!put(c, q) && !devices::live.count(q));
  devices::refuse = false;
  REQUIRE(!c.put(nullptr, false) && c.put(nullptr, true));
  put(c, hold);
  REQUIRE(devices::live.empty());
}

// The object of one device is destroyed while the library works on another,
// from a thread on either
void two_devices()
{
  for (int from = 0; from < 2; from++) {
    cache_t c;
    devices::now = 0;
    void *a = take(c, 20 * MB);
    devices::now = 1;
    void *b = take(c, 1000);
    devices::now = from;
    put(c, a);
    REQUIRE(c.kept_bytes(1) == 0);
    devices::now = 1;
    void *d = take(c, 20 * MB); // take checks its device
    REQUIRE(d != a);
    devices::now = 0;
    if (from == 0) REQUIRE(take(c, 20 * MB) == a); // kept where it belongs
    if (from == 0) put(c, a);
    devices::now = 1;
    put(c, d);
    put(c, b);
    REQUIRE(devices::live.empty());
  }
  devices::now = 0;
}

void limits()
{
  cache_t c;
  void *hold = take(c, 1000);
  std::vector<void *> many;
  for (int i = 0; i < 12; i++) many.push_back(take(c, 700 * MB));
  for (void *p : many) put(c, p);
  REQUIRE(c.kept_bytes(0) <= mfp::CACHE_BYTES);
  REQUIRE(c.kept_bytes(0) >= mfp::CACHE_BYTES - 1024 * MB);
  // the latest are kept, the first ones made room
  REQUIRE(!devices::live.count(many[0]) && devices::live.count(many[11]));
  std::vector<void *> small;
  for (int i = 0; i < 100; i++) small.push_back(take(c, 50 * MB));
  for (void *p : small) put(c, p);
  REQUIRE(c.kept_bytes(0) <= mfp::CACHE_BYTES && !devices::live.count(many[11]) && devices::live.count(small[99]));
  // an allocation that fails takes back what is kept, the caller's own too
  devices::limit = devices::bytes + MB;
  void *big = take(c, 900 * MB);
  REQUIRE(c.kept_bytes(0) == 0);
  void *own = nullptr;
  put(c, big);
  REQUIRE(c.alloc(&own, 3800 * MB));
  REQUIRE(c.kept_bytes(0) == 0);
  devices::release(own);
  // exactly the last bytes: without the rounding to a class
  devices::limit = devices::bytes + 70001;
  void *tight = c.get(70001);
  REQUIRE(tight && devices::live[tight].size == 70001);
  REQUIRE(!c.get(70001));
  put(c, tight);
  devices::limit = ~size_t(0);
  // a device that cannot be waited for keeps nothing
  void *p = take(c, 10 * MB);
  devices::free_fails = true;
  put(c, p);
  devices::free_fails = false;
  REQUIRE(c.kept_bytes(0) == 0 && !devices::live.count(p));
  put(c, hold);
  put(c, nullptr);
  REQUIRE(devices::live.empty());
}

void threads()
{
  cache_t c;
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; t++)
    ts.emplace_back([&c, t] {
      std::mt19937 rng(t);
      std::vector<void *> held;
      for (int i = 0; i < 4000; i++) {
        devices::now = (int)(rng() % 2);
        if (held.size() < 6 && rng() % 2) {
          held.push_back(take(c, 1 + (size_t)(rng() % 4 ? rng() % (2 * MB) : rng() % (80 * MB))));
        } else if (!held.empty()) {
          const size_t k = rng() % held.size();
          put(c, held[k]); // from either device
          held[k] = held.back();
          held.pop_back();
        }
        if (rng() % 500 == 0) c.trim();
      }
      for (void *p : held) put(c, p);
    });
  for (auto &t : ts) t.join();
  REQUIRE(devices::live.empty() && devices::bytes == 0);
}

} // namespace

int main()
{
  reuse();
  refused();
  together();
  two_devices();
  limits();
  threads();
  std::printf("ALL OK\n");
}
