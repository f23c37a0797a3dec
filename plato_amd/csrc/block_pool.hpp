// The device blocks of a context: which there are, and those kept for reuse after they were
// freed.  Host code only: it hands addresses out and takes them back, dmalloc and dfree
// allocate and free them.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>

namespace pe {

// Device blocks that a context keeps after they are freed, for its next allocations of about
// the same size: an algorithm's scratch is allocated and freed by every call, and a hipFree
// waits for the device (BFS scale 24, 14 blocks of 0.5 GB in all: 5.2 ms a call without, 2.7 ms
// with; nine engine calls at scale 12: 0.56 and 0.32 ms).  Bounded by POOL_BYTES, the blocks
// kept longest leaving first; given back when an allocation of any context on the device fails,
// when the caller asks for it, and when the context goes.
// All work of a context is on one stream, so a block's next user runs after its last one.
// Every member may be called from several threads: a context's calls come from one at a time,
// but its objects may be destroyed by another meanwhile (a garbage collector's).
class block_pool {
 public:
  static constexpr size_t POOL_BYTES = 1ull << 30, BLOCK_BYTES = 512ull << 20;

  // the size of the block that serves a request of `bytes`: whole units of 512, as far as size_t goes
  static size_t block_size(size_t bytes) {
    return bytes > SIZE_MAX - 511 ? bytes : (std::max<size_t>(bytes, 1) + 511) & ~(size_t)511;
  }

  // a kept block of `want` to a quarter more bytes, or nullptr
  void* take(size_t want) {
    std::lock_guard<std::mutex> lock(mu);
    auto it = kept.lower_bound(want);
    if (it == kept.end() || it->first - want > want / 4) return nullptr;
    void* p = it->second.p;
    kept_total -= it->first;
    kept.erase(it);
    return p;
  }

  // a new block; may throw (no host memory), and then it is not one of the pool's
  void add(void* p, size_t size) {
    std::lock_guard<std::mutex> lock(mu);
    size_of.emplace(p, size);
  }

  // A block that its owner is done with: kept, or, when true is returned, for the caller to free.
  bool give(void* p) noexcept {
    std::lock_guard<std::mutex> lock(mu);
    auto it = size_of.find(p);
    if (it == size_of.end()) return false;
    const size_t size = it->second;
    if (size <= BLOCK_BYTES) {
      try {
        kept.emplace(size, entry{p, ++clock});
        kept_total += size;
        return false;
      } catch (...) {  // no host memory for the entry
      }
    }
    size_of.erase(it);
    return true;
  }

  // the block kept longest while more than `bound` bytes are kept, for the caller to free; or nullptr
  void* oldest_over(size_t bound) noexcept {
    std::lock_guard<std::mutex> lock(mu);
    if (kept_total <= bound) return nullptr;
    auto old = std::min_element(kept.begin(), kept.end(),
                                [](const auto& x, const auto& y) { return x.second.age < y.second.age; });
    void* p = old->second.p;
    size_of.erase(p);
    kept_total -= old->first;
    kept.erase(old);
    return p;
  }

  size_t kept_bytes() const {
    std::lock_guard<std::mutex> lock(mu);
    return kept_total;
  }

  // bytes asked for by the blocks in use
  void charge(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    used += bytes;
  }
  void credit(size_t bytes) noexcept {
    std::lock_guard<std::mutex> lock(mu);
    used -= bytes;
  }
  uint64_t used_bytes() const {
    std::lock_guard<std::mutex> lock(mu);
    return used;
  }

 private:
  struct entry {
    void* p;
    uint64_t age;
  };
  mutable std::mutex mu;
  std::multimap<size_t, entry> kept;          // free blocks by size
  std::unordered_map<void*, size_t> size_of;  // every block of the context
  uint64_t clock = 0;
  size_t kept_total = 0;
  uint64_t used = 0;
};

}  // namespace pe
