// Released device blocks kept for the next allocation (no GPU header: the
// allocator underneath is a parameter).
//
// hipMalloc + hipFree take 0.1-0.3 ms a pair here and hipFree waits for the
// device: the 35 temporaries of one 64^3-hexahedra assembly took 5.9 of its 7.8
// ms.  Every block is used on the library's one stream (the upload streams wait
// for it first), so a block handed on while earlier work is still enqueued is
// safe by stream order, from any thread.  At most `limit` bytes stay cached; past
// that the largest go back at once.  Blocks of other devices than the first one
// used are never kept.
#pragma once

#include <cstddef>
#include <iterator>
#include <map>
#include <mutex>

namespace mh {

// Size class of an allocation, so that blocks fit one another's requests: steps
// of an eighth of the leading power of two.
inline size_t pool_round(size_t bytes) {
  size_t step = 512;
  while (step * 16 <= bytes) step <<= 1;
  return (bytes + step - 1) / step * step;
}

// Sys: `bool alloc(void** p, size_t bytes)` and `void free(void* p)`.
template <class Sys>
class BlockPool {
 public:
  explicit BlockPool(size_t limit, Sys sys = Sys()) : limit_(limit), sys_(sys) {}

  // A block of at least `bytes` on device `dev` (the current one); *cap is handed
  // back to free.  A request that the memory does not hold beside the cached blocks
  // gets them all freed, and what fits exactly is not refused for its rounding.
  bool alloc(void** p, size_t bytes, int dev, size_t* cap) {
    const size_t want = bytes;
    bytes = pool_round(bytes);
    bool own = false;
    {
      std::lock_guard<std::mutex> lk(mu_);
      if (device_ < 0) device_ = dev;
      own = dev == device_ && bytes <= limit_;
      if (own) {
        auto it = blocks_.lower_bound(bytes);
        if (it != blocks_.end() && it->first <= bytes + bytes / 4) {
          *p = it->second;
          *cap = it->first;
          cached_ -= it->first;
          blocks_.erase(it);
          return true;
        }
      }
    }
    *cap = own ? bytes : 0;  // 0: freed at once
    if (alloc_outside(p, own ? bytes : want)) return true;
    *cap = 0;
    return own && sys_.alloc(p, want);
  }

  // Called from destructors: nothing thrown leaves it.
  void free(void* p, size_t cap) {
    if (!p) return;
    bool kept = false;
    if (cap > 0 && cap <= limit_) {
      try {
        std::lock_guard<std::mutex> lk(mu_);
        blocks_.emplace(cap, p);
        cached_ += cap;
        kept = true;
      } catch (...) {
      }
    }
    if (!kept) sys_.free(p);
    for (;;) {
      void* q = nullptr;
      {
        std::lock_guard<std::mutex> lk(mu_);
        if (cached_ <= limit_) break;
        auto it = std::prev(blocks_.end());
        cached_ -= it->first;
        q = it->second;
        blocks_.erase(it);
      }
      sys_.free(q);
    }
  }

  // Memory that is not the pool's (user buffers), which may need what the pool holds.
  bool alloc_outside(void** p, size_t bytes) {
    if (sys_.alloc(p, bytes)) return true;
    return trim() > 0 && sys_.alloc(p, bytes);
  }

  // Frees every cached block; returns their bytes.
  size_t trim() {
    std::multimap<size_t, void*> old;
    size_t bytes = 0;
    {
      std::lock_guard<std::mutex> lk(mu_);
      old.swap(blocks_);
      bytes = cached_;
      cached_ = 0;
    }
    for (auto& q : old) sys_.free(q.second);
    return bytes;
  }

 private:
  size_t limit_;
  Sys sys_;
  std::mutex mu_;
  std::multimap<size_t, void*> blocks_;  // by size
  size_t cached_ = 0;
  int device_ = -1;
};

}  // namespace mh
