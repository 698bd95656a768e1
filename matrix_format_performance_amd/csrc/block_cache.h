// Freed device blocks, kept for the library's next allocations.  Host code
// only; the device calls come from Dev, so that the bookkeeping can be checked
// without a GPU:
//   static bool alloc(void **p, size_t bytes)  on the current device; of no
//                                              bytes: whether it may be called
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
//  * A block is kept once its device is idle: by put, which waits as hipFree
//    does, or by its caller's word (a stream that was waited for and alone used
//    it). Whoever gets it next, on any stream or thread, finds nothing still
//    running on it.  put waits by freeing a token, a small allocation that it
//    makes for that: hipDeviceSynchronize would wait as well, but it ends every
//    stream capture in the process, also those that another thread's hipFree
//    leaves alone.
//  * get is refused where hipMalloc is, in a stream capture, also when a kept
//    block would do: an allocation of no bytes asks.
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
        void *none = nullptr;
        if (Dev::alloc(&none, 0)) {
          std::lock_guard<std::mutex> lock(mutex_);
          taken(p, b);
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
    taken(p, b);
    return p;
  }

  // Gives back a block of get.  idle: nothing still uses it.  Returns idle, or
  // that the current device was waited for.
  bool put(void *p, bool idle)
  {
    if (!p) return idle;
    block b{-1, 0};
    {
      std::lock_guard<std::mutex> lock(mutex_);
      const auto it = sizes_.find(p);
      if (it != sizes_.end()) {
        b = it->second;
        sizes_.erase(it);
      }
    }
    // waiting is for the current device, so only its blocks are kept
    const bool own = b.second && Dev::current() == b.first;
    if (own && !idle) {
      void *token = nullptr;
      idle = Dev::alloc(&token, TOKEN) && Dev::release(token);
    }
    blocks out;
    if (!(own && idle && add(b, p, out))) (void)Dev::release(p);
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (--in_use_ == 0) {
        out.merge(kept_);
        kept_bytes_ = 0;
      }
    }
    release(out);
    return idle;
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
  void taken(void *p, const block &b)
  {
    in_use_++;
    try {
      if (b.second) sizes_[p] = b;
    } catch (const std::bad_alloc &) {
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
  std::unordered_map<void *, block> sizes_; // cacheable blocks in use
  size_t kept_bytes_ = 0;
  uint64_t puts_ = 0;
  size_t in_use_ = 0; // blocks of any size
};

} // namespace mfp
