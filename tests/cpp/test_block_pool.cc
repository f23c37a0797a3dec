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

int main() {
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
