// Transfers between device memory and ordinary (pageable) host memory through a small ring of
// pinned slots.
//
// The runtime's own pageable copies stage on one thread, and a result array that the caller
// has just allocated takes a page fault per touched page on that thread too: 10.6 GB/s into
// fresh memory, 17.6 GB/s into warm, 29.6 GB/s from host, against 57 GB/s of the link.  Here a
// chunk goes to a pinned slot (copied, or written there by a kernel that reorders it on the
// way, so no device-side copy of the result is needed) while worker threads move earlier
// chunks on.  The ring belongs to the context (16 MiB, made by the first transfer, freed with
// it); the threads live for one call.
// PageRank RMAT scale 26, 20 iterations, with its 512 MB result (256 MB over the link, widened
// by the workers): 137 -> 50 ms; BFS scale 24 with its 64 MB of levels 9.8 -> 5.1 ms.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

#include "pe_internal.hpp"

namespace pe {

static constexpr int ST_SLOTS = 8;
static constexpr size_t ST_BYTES = 2u << 20;      // per slot
static constexpr unsigned ST_THREADS = 6;         // workers at most
static constexpr uint64_t ST_INLINE_CHUNKS = 3;   // up to this many the calling thread moves alone
// A worker polls for its chunk a while and then sleeps between looks: the next chunk of a running
// transfer is there within 40 us, but the work queued before the first may take any time (300 ms
// of it, CPU time of the process: 2.0 s polling, 0.32 s so).
static constexpr int ST_POLLS = 10000;
static constexpr int ST_SLEEP_US = 100;
static constexpr size_t ST_SMALL = 256u << 10;    // the runtime's own copy is as fast up to here; up to
                                                  // MAIL_WORDS words come by mail (nine engine calls and
                                                  // two results of 16 KB: 312 -> 239 us with theirs)

struct staging {
  uint8_t* ring = nullptr;
  hipEvent_t ev[ST_SLOTS] = {};
  uint8_t* slot(uint64_t c) const { return ring + (c % ST_SLOTS) * ST_BYTES; }
  ~staging() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (ring) (void)hipHostFree(ring);
  }
};

void staging_free(staging* st) { delete st; }

static staging& ring_of(pe_ctx_s* ctx) {
  if (!ctx->stage) {
    auto st = std::make_unique<staging>();
    PE_HIP(hipHostMalloc(reinterpret_cast<void**>(&st->ring), ST_SLOTS * ST_BYTES, hipHostMallocDefault));
    for (hipEvent_t& e : st->ev) PE_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    ctx->stage = st.release();
  }
  return *ctx->stage;
}

namespace {

// Workers that take chunks in order: each waits until its chunk may be moved (`ready`), moves
// it and marks it.  Joined by the destructor, which also ends them early when the calling
// thread leaves by an exception.
struct workers {
  std::atomic<uint64_t> ready{0}, next{0};
  std::atomic<bool> stop{false};
  std::vector<std::atomic<uint8_t>> done;
  std::vector<std::thread> threads;
  uint64_t chunks;

  template <typename F>
  workers(uint64_t n, const F& move) : done(n), chunks(n) {
    const unsigned want = n <= ST_INLINE_CHUNKS
                              ? 0u
                              : (unsigned)std::min<uint64_t>({ST_THREADS, n / 2, std::max(1u, std::thread::hardware_concurrency())});
    try {
      threads.reserve(want);
      for (unsigned t = 0; t < want; ++t)
        threads.emplace_back([this, move] {
          for (;;) {
            const uint64_t c = next.fetch_add(1);
            if (c >= chunks) return;
            for (int k = 0; ready.load(std::memory_order_acquire) <= c; ++k) {
              if (stop.load(std::memory_order_relaxed)) return;
              if (k < ST_POLLS) std::this_thread::yield();
              else std::this_thread::sleep_for(std::chrono::microseconds(ST_SLEEP_US));
            }
            move(c);
            done[c].store(1, std::memory_order_release);
          }
        });
    } catch (...) {
      // no (more) threads: those that started, or the calling thread, do it all
    }
  }
  ~workers() {
    stop.store(true);
    for (auto& t : threads) t.join();
  }
  bool moved(uint64_t c) const { return done[c].load(std::memory_order_acquire) != 0; }
};

}  // namespace

void staged_download(pe_ctx_s* ctx, uint64_t units, size_t unit_bytes, const stage_fn& launch, const stage_fn& consume) {
  if (!units) return;
  staging& st = ring_of(ctx);
  hipStream_t s = ctx->stream;
  const uint64_t per = std::max<uint64_t>(1, ST_BYTES / unit_bytes), n = (units + per - 1) / per;
  if (n == 1) {
    launch(0, units, st.slot(0));
    PE_HIP(hipStreamSynchronize(s));
    consume(0, units, st.slot(0));
    return;
  }
  auto move = [&, per, units](uint64_t c) { consume(c * per, std::min(per, units - c * per), st.slot(c)); };
  workers w(n, move);
  uint64_t issued = 0, ready = 0;
  while (ready < n) {
    while (issued < n && issued - ready < ST_SLOTS && (issued < ST_SLOTS || w.moved(issued - ST_SLOTS))) {
      launch(issued * per, std::min(per, units - issued * per), st.slot(issued));
      PE_HIP(hipEventRecord(st.ev[issued % ST_SLOTS], s));
      ++issued;
    }
    if (ready == issued) {  // the workers have every slot
      std::this_thread::yield();
      continue;
    }
    PE_HIP(hipEventSynchronize(st.ev[ready % ST_SLOTS]));
    if (w.threads.empty()) {
      move(ready);
      w.done[ready].store(1, std::memory_order_release);
    }
    w.ready.store(++ready, std::memory_order_release);
  }
  for (uint64_t c = n > ST_SLOTS ? n - ST_SLOTS : 0; c < n; ++c)  // earlier ones were waited for
    while (!w.moved(c)) std::this_thread::yield();
}

void host_download(pe_ctx_s* ctx, const void* dev, void* host, size_t bytes) {
  if (bytes && bytes <= MAIL_WORDS * 4 && bytes % 4 == 0) {
    std::memcpy(host, mail_words(ctx, static_cast<const uint32_t*>(dev), (uint32_t)(bytes / 4)), bytes);
    return;
  }
  if (bytes <= ST_SMALL) {
    if (bytes) PE_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, ctx->stream));
    PE_HIP(hipStreamSynchronize(ctx->stream));
    return;
  }
  staged_download(
      ctx, bytes, 1,
      [&](uint64_t u0, uint64_t n, void* slot) {
        PE_HIP(hipMemcpyAsync(slot, static_cast<const uint8_t*>(dev) + u0, n, hipMemcpyDeviceToHost, ctx->stream));
      },
      [&](uint64_t u0, uint64_t n, void* slot) { std::memcpy(static_cast<uint8_t*>(host) + u0, slot, n); });
}

void host_upload(pe_ctx_s* ctx, void* dev, const void* host, size_t bytes) {
  hipStream_t s = ctx->stream;
  if (bytes <= ST_SMALL) {
    if (bytes) PE_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s));
    PE_HIP(hipStreamSynchronize(s));
    return;
  }
  staging& st = ring_of(ctx);
  const uint64_t n = (bytes + ST_BYTES - 1) / ST_BYTES;
  auto move = [&, bytes](uint64_t c) {
    std::memcpy(st.slot(c), static_cast<const uint8_t*>(host) + c * ST_BYTES,
                std::min<size_t>(ST_BYTES, bytes - c * ST_BYTES));
  };
  workers w(n, move);
  // half of the ring is being filled while the other half is on its way
  constexpr uint64_t HALF = ST_SLOTS / 2;
  w.ready.store(std::min<uint64_t>(n, ST_SLOTS), std::memory_order_release);
  for (uint64_t c = 0; c < n; ++c) {
    if (c >= HALF) {
      PE_HIP(hipEventSynchronize(st.ev[(c - HALF) % ST_SLOTS]));
      w.ready.store(std::min<uint64_t>(n, c - HALF + 1 + ST_SLOTS), std::memory_order_release);
    }
    if (w.threads.empty()) move(c);
    else
      while (!w.moved(c)) std::this_thread::yield();
    PE_HIP(hipMemcpyAsync(static_cast<uint8_t*>(dev) + c * ST_BYTES, st.slot(c),
                          std::min<size_t>(ST_BYTES, bytes - c * ST_BYTES), hipMemcpyHostToDevice, s));
    PE_HIP(hipEventRecord(st.ev[c % ST_SLOTS], s));
  }
  PE_HIP(hipStreamSynchronize(s));  // the slots are free for the next transfer
}

}  // namespace pe
