// The block pool of a context under several threads, with plain memory in place of the
// device's: every block has one owner at a time, what is kept stays within the bound, and all
// of it comes back at the end.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#include "block_pool.hpp"

static pe::block_pool pool;
static std::atomic<long> live{0};

static void release(void* p) {
  std::free(p);
  --live;
}

// a request near the largest size_t keeps its size (a multiple of 512 would wrap to nothing) and
// is served by no smaller block that is kept
static int wrong_sizes() {
  int bad = 0;
  for (size_t bytes : {(size_t)0, (size_t)1, (size_t)511, (size_t)512, (size_t)513, (size_t)1 << 40})
    bad += pe::block_pool::block_size(bytes) % 512 != 0 || pe::block_pool::block_size(bytes) < std::max<size_t>(bytes, 1);
  pe::block_pool p;
  void* small = &bad;
  p.add(small, 512);
  bad += p.give(small);
  for (size_t off : {0, 7, 510, 511, 512, 1000}) {
    const size_t bytes = SIZE_MAX - off;
    bad += pe::block_pool::block_size(bytes) < bytes;
    bad += p.take(pe::block_pool::block_size(bytes)) != nullptr;
  }
  return bad;
}

int main() {
  if (int n = wrong_sizes()) {
    std::printf("wrong sizes: %d\n", n);
    return 1;
  }
  constexpr int THREADS = 4, ROUNDS = 20000;
  std::atomic<int> bad{0};
  auto work = [&](unsigned id) {
    std::mt19937 rng(id);
    std::vector<std::pair<unsigned*, size_t>> mine;
    for (int i = 0; i < ROUNDS; ++i) {
      if (mine.size() < 8 && rng() % 2) {
        const size_t bytes = 1 + rng() % 5000, want = pe::block_pool::block_size(bytes);
        void* p = pool.take(want);
        if (!p) {
          p = std::malloc(want);
          ++live;
          pool.add(p, want);
        }
        pool.charge(bytes);
        *static_cast<unsigned*>(p) = id;
        mine.emplace_back(static_cast<unsigned*>(p), bytes);
      } else if (!mine.empty()) {
        const size_t k = rng() % mine.size();
        auto [p, bytes] = mine[k];
        mine[k] = mine.back();
        mine.pop_back();
        if (*p != id) ++bad;  // someone else holds it too
        pool.credit(bytes);
        if (pool.give(p)) release(p);
        while (void* old = pool.oldest_over(1 << 16)) release(old);
        (void)pool.kept_bytes();
      }
    }
    for (auto [p, bytes] : mine) {
      pool.credit(bytes);
      if (pool.give(p)) release(p);
    }
  };
  std::vector<std::thread> threads;
  for (int t = 0; t < THREADS; ++t) threads.emplace_back(work, 100u + t);
  for (auto& t : threads) t.join();
  while (void* p = pool.oldest_over(0)) release(p);
  std::printf("shared blocks: %d, left: %ld, kept: %zu, used: %llu\n", bad.load(), live.load(), pool.kept_bytes(),
              (unsigned long long)pool.used_bytes());
  return bad || live || pool.kept_bytes() || pool.used_bytes() ? 1 : 0;
}
