// Freed device blocks, kept for the library's next allocations.  Host code
// only; the device calls come from Dev, so that the bookkeeping can be checked
// without a GPU:
//   static bool alloc(void **p, size_t bytes)  on the current device
//   static bool release(void *p)               of any device; waits for the current one
//   static int current()                       the current device, -1 unknown
#pragma once

#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <new>
#include <unordered_map>
#include <utility>

namespace mfp {

// hipMalloc / hipFree map and unmap memory: 30 to 90 us per call for blocks of
// 16 MB and more, 210 to 250 us to free one while others are held, so that
// building one plan spent more on its ten or so arrays than on its kernels
// (nine formats of a 5M-entry matrix: 1.8 ms of kernels in 8.7 to 12.9 ms).
// Freed blocks of 64 KB to 1 GB are therefore kept and handed out again, in
// size classes an eighth of a power of two apart.
//  * Every block that is taken from the cache or put there goes with a token, a
//    small allocation of its own (1.4 us to allocate and free).  Allocating it
//    is refused where hipMalloc is, in a stream capture; freeing it waits for the
//    device as hipFree does, so that whoever gets the block next, on any stream
//    or thread, finds nothing still running on it.  hipDeviceSynchronize (0.2 us
//    on an idle device) would wait as well, but it ends every stream capture in
//    the process, also those that another thread's hipFree leaves alone.
//  * A block is filed under the device it was allocated on, whichever device
//    the freeing thread uses, and handed out on that device only.
//  * At most CACHE_BYTES are kept, the oldest make room; an allocation that
//    fails gives all of them back and tries again, and they are given back by
//    trim and when the library's last block is freed.
constexpr size_t CACHE_MIN = 64u << 10, CACHE_MAX = 1u << 30, CACHE_BYTES = 4ull << 30;

template <class Dev>
class block_cache {
  using block = std::pair<int, size_t>; // device, size (0: not cacheable)
  struct kept {
    void *p;
    uint64_t since; // counts the blocks that were put
  };
  using blocks = std::multimap<block, kept>;
  struct held {
    block b;
    void *token;
  };
  static constexpr size_t TOKEN = 256;

public:
  // a block of at least bytes on the current device, null when there is none
  void *get(size_t bytes)
  {
    const int device = Dev::current();
    const bool cacheable = bytes >= CACHE_MIN && bytes <= CACHE_MAX && device >= 0;
    const size_t size = cacheable ? size_class(bytes) : bytes;
    if (cacheable) {
      block b{-1, 0};
      if (void *p = take_kept(device, size, b)) {
        void *token = nullptr;
        if (Dev::alloc(&token, TOKEN)) {
          std::lock_guard<std::mutex> lock(mutex_);
          taken(p, b, token);
          return p;
        }
        (void)Dev::release(p);
      }
    }
    void *p = nullptr;
    block b{device, cacheable ? size : 0};
    if (!alloc(&p, size)) {
      b.second = 0;
      if (size == bytes || !Dev::alloc(&p, bytes)) return nullptr; // without the rounding, then
    }
    std::lock_guard<std::mutex> lock(mutex_);
    taken(p, b, nullptr);
    return p;
  }

  // gives back a block of get
  void put(void *p)
  {
    if (!p) return;
    held h{{-1, 0}, nullptr};
    {
      std::lock_guard<std::mutex> lock(mutex_);
      const auto it = sizes_.find(p);
      if (it != sizes_.end()) {
        h = it->second;
        sizes_.erase(it);
      }
    }
    // freeing waits for the current device, so only its blocks are kept
    const bool own = h.b.second && Dev::current() == h.b.first;
    if (own && !h.token && !Dev::alloc(&h.token, TOKEN)) h.token = nullptr;
    const bool idle = h.token && Dev::release(h.token) && own;
    blocks out;
    if (!(idle && add(h.b, p, out))) (void)Dev::release(p);
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (--in_use_ == 0) {
        out.merge(kept_);
        kept_bytes_ = 0;
      }
    }
    release(out);
  }

  // an allocation beside the cache's own that may take what it keeps
  bool alloc(void **p, size_t bytes)
  {
    if (Dev::alloc(p, bytes)) return true;
    trim();
    return Dev::alloc(p, bytes);
  }

  // gives back every kept block
  void trim()
  {
    blocks out;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      out.swap(kept_);
      kept_bytes_ = 0;
    }
    release(out);
  }

  // bytes kept on a device
  size_t kept_bytes(int device)
  {
    std::lock_guard<std::mutex> lock(mutex_);
    size_t sum = 0;
    for (auto it = kept_.lower_bound({device, 0}); it != kept_.end() && it->first.first == device; ++it)
      sum += it->first.second;
    return sum;
  }

private:
  static size_t size_class(size_t bytes)
  {
    size_t step = CACHE_MIN / 8;
    while (step * 16 <= bytes) step *= 2; // 8 step <= bytes < 16 step
    return (bytes + step - 1) / step * step;
  }

  // the smallest kept block that will do, null when there is none
  void *take_kept(int device, size_t size, block &b)
  {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto it = kept_.lower_bound({device, size});
    if (it == kept_.end() || it->first.first != device || it->first.second > size + size / 4) return nullptr;
    void *p = it->second.p;
    b = it->first;
    kept_bytes_ -= b.second;
    kept_.erase(it);
    return p;
  }

  // mutex_ held; without memory for the entry the block is not cacheable
  void taken(void *p, const block &b, void *token)
  {
    in_use_++;
    try {
      if (b.second) sizes_[p] = held{b, token};
    } catch (const std::bad_alloc &) {
      if (token) (void)Dev::release(token);
    }
  }

  // the blocks that make room for it go to out
  bool add(const block &b, void *p, blocks &out)
  {
    std::lock_guard<std::mutex> lock(mutex_);
    typename blocks::iterator at;
    try {
      at = kept_.emplace(b, kept{p, ++puts_});
    } catch (const std::bad_alloc &) {
      return false;
    }
    kept_bytes_ += b.second;
    while (kept_bytes_ > CACHE_BYTES) { // CACHE_MAX is below it: not the new one
      auto oldest = at;
      for (auto it = kept_.begin(); it != kept_.end(); ++it)
        if (it->second.since < oldest->second.since) oldest = it;
      kept_bytes_ -= oldest->first.second;
      out.insert(kept_.extract(oldest));
    }
    return true;
  }

  // without the mutex: giving memory back takes its time
  static void release(const blocks &out)
  {
    for (const auto &b : out) (void)Dev::release(b.second.p);
  }

  std::mutex mutex_;
  blocks kept_;
  std::unordered_map<void *, held> sizes_; // cacheable blocks in use
  size_t kept_bytes_ = 0;
  uint64_t puts_ = 0;
  size_t in_use_ = 0; // blocks of any size
};

} // namespace mfp
