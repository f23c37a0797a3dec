// k-core decomposition: plato::algo::kcore_algo_t::compute_shell_index
// (plato/algo/kcore/kcore.hpp:80-268) on the device.
//
// The reference iterates the h-index operator of Montresor et al. (IEEE TPDS 2012)
// synchronously: coreness starts at the adjacency length (0xFFFFFFFF for vertices
// without one), every vertex is active in epoch 0, and in each epoch every active
// vertex v with est = min(len(v), estimate[v]) takes the largest i in [1, est] such
// that at least i neighbours u have min(est, estimate[u]) >= i, when that i is below
// its coreness (v is then modified and its neighbours become active for the next
// epoch); a vertex with no neighbours gets 0; when no i qualifies the value is kept.
// Estimates are the previous epoch's values (Jacobi), so the result and the per-epoch
// counts do not depend on the order of the vertices: they are compared bit for bit
// with the oracle.
//
// On a symmetrized graph the adjacency is its own reverse, and most active vertices keep
// their value, so the device carries cnt(v) = the neighbours u with estimate[u] >=
// estimate[v] along with the estimates: v is modified in an epoch exactly when cnt(v) <
// estimate[v].  A vertex that drops from `old` to `now` takes one from cnt(u) of every
// unmodified neighbour u with now < estimate[u] <= old and re-counts its own, so an epoch
// reads the adjacencies of the modified vertices instead of those of all active ones, twice
// where a vertex is newly modified and once where it was in the epoch before; the active set
// is still marked and counted, for the per-epoch log.  In epoch 0 everything is active; a vertex
// that keeps its adjacency length has cnt(v) equal to it.
// RMAT scale 22 symmetrized, degree-relabeled, 38 epochs, whole call: 51 ms re-counting every
// active vertex, 20 ms with the counts, 16.1 ms with the drops found in the spread before,
// 15.6 ms with the marks in the values.  Bound by the rate of the random 4-byte reads of the
// values in the first ten epochs, when most vertices are modified (1.2 ms per walk of the 2^27
// entries, 112 G/s; twice as many in flight per lane: 16.3 ms).
// Other adjacencies (in-edges or out-edges of a directed graph) have no counts: every
// active vertex is re-counted.
//
// Per epoch: the candidate bitmap (vertices with cnt < estimate; the active set without
// counts) is cut into queues by adjacency length, then
//   h-index:  one lane per vertex of at most KC_SMALL neighbours (byte histogram of its own
//             in LDS), one wave up to KC_HUGE when the answer cannot exceed KC_HIST (KC_HIST
//             + 1 LDS bins per wave), one 1024-thread block up to KC_GIANT, and chunks over
//             all blocks beyond (their histograms add up in global memory); answers above
//             KC_HHIST take a histogram of value ranges first and one of the range's values
//             next, each halving the candidates' bits by 14;
//   spread:   modified vertices activate their neighbours and update the counts;
//   commit:   estimate = coreness, next epoch's candidates and the log's counters, which
//             reach the host in one mail.
#include <algorithm>
#include <vector>

#include "pe_internal.hpp"

namespace pe {

static constexpr uint32_t KC_UNSET = 0xFFFFFFFFu;
// A count with this bit is none: the vertex falls short, and the other bits are its value of the
// next epoch (of a vertex of at most KC_GIANT neighbours).  Counts of more than 2^31 neighbours
// have the bit too, which at most makes such a vertex a candidate that keeps its value.
static constexpr uint32_t KC_AHEAD = 0x80000000u;
static constexpr uint32_t KC_SMALL = 64;    // neighbours handled by one lane
static constexpr uint32_t KC_HIST = 1024;   // histogram bins 0..KC_HIST of the wave-per-vertex pass
static constexpr uint32_t KC_PER = 17;      // bins per lane in its scan (64 * 17 > KC_HIST)
static constexpr int KC_THREADS = 256;
static constexpr uint32_t KC_HUGE = 4096;    // longer adjacencies take one block each
static constexpr int KC_HTHREADS = 1024;
static constexpr uint32_t KC_HBITS = 14;
static constexpr uint32_t KC_HHIST = 1u << KC_HBITS;  // histogram bins 0..KC_HHIST of the block pass
static constexpr uint32_t KC_HPER = 17;      // bins per thread in its scan (1024 * 17 > KC_HHIST)
static constexpr uint64_t KC_GIANT = 65536;  // longer adjacencies are cut into chunks over many blocks
static constexpr uint64_t KC_GCHUNK = 16384;
static constexpr int KC_U = 4;               // neighbours a lane of the wave and block passes has in flight
static_assert(64 * (KC_SMALL + 1) <= 64 * KC_PER * 4, "a wave's byte histograms fit in the space of its bins");

struct kc_counters {
  unsigned long long nsmall, nbig, nhuge;  // queued candidates by adjacency length
  unsigned long long modified;             // vertices whose coreness dropped
  unsigned long long next_active;          // size of the next active set
  unsigned long long next_cand;            // candidates of the next epoch
  unsigned long long giant_top;            // largest estimate among the giants re-counted in this epoch
};
static constexpr uint32_t KC_CW = sizeof(kc_counters) / 8;

// where a giant's h-index stands between two histogram rounds: it lies in the bins base +
// [j << shift, (j + 1) << shift), j <= nb, of the round to come, with `above` neighbours over
// them; shift -1: done
struct kc_giant {
  uint32_t base, above, nb;
  int32_t shift;
};

__global__ void k_kc_init(const uint64_t* __restrict__ ptr, uint32_t V, uint32_t* __restrict__ core,
                          uint32_t* __restrict__ est, uint32_t* __restrict__ cnt) {
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t len = ptr[v + 1] - ptr[v];
    const uint32_t c = len ? (uint32_t)std::min<uint64_t>(len, 0xFFFFFFFEull) : KC_UNSET;
    core[v] = c;
    est[v] = c;
    if (cnt) cnt[v] = len ? c : 0u;
  }
}

__global__ void k_kc_fill(uint64_t* __restrict__ w, uint64_t nwords, uint32_t V) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < nwords; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t lo = i * 64;
    uint64_t m = 0ull;
    if (lo + 64 <= V) m = ~0ull;
    else if (lo < V) m = (1ull << (V - lo)) - 1ull;
    w[i] = m;
  }
}

__global__ void k_kc_zero(uint64_t* __restrict__ w, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    w[i] = 0ull;
}

// the reference's `if (!get_bit(u)) set_bit(u)`
__device__ __forceinline__ void kc_set_bit(uint64_t* bits, uint32_t u) {
  const uint64_t m = 1ull << (u & 63);
  if (!(bits[u >> 6] & m)) atomicOr((unsigned long long*)&bits[u >> 6], (unsigned long long)m);
}

// ---- queues ------------------------------------------------------------------------------
// Candidate bitmap -> queues by adjacency length, the bitmap cleared for the next epoch's
// marks.  One wave per word, lane = bit, so the offsets are read coalesced; a block takes 64
// words at a time and reserves its slots of the three queues with one atomic each.  Giants
// go to no queue: their bits are kept in `act` (nullptr without giants).
static constexpr int KC_CW_WORDS = 4;  // words per wave and step
__global__ __launch_bounds__(1024) void k_kc_classify(uint64_t* __restrict__ cand, uint64_t* __restrict__ act,
                                                      uint64_t nwords, uint32_t V, const uint64_t* __restrict__ ptr,
                                                      const uint32_t* __restrict__ est, uint32_t* __restrict__ qsmall,
                                                      uint32_t* __restrict__ qbig, uint32_t* __restrict__ qhuge_end,
                                                      kc_counters* __restrict__ cnt) {
  __shared__ uint32_t s_cnt[3][16];
  __shared__ unsigned long long s_base[3];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  constexpr uint64_t STEP = 16 * KC_CW_WORDS;
  for (uint64_t w0 = blockIdx.x * STEP; w0 < nwords; w0 += (uint64_t)gridDim.x * STEP) {
    uint64_t m[3][KC_CW_WORDS];
    uint32_t n[3] = {0, 0, 0};
#pragma unroll
    for (int j = 0; j < KC_CW_WORDS; ++j) {
      const uint64_t word = w0 + (uint64_t)wave * KC_CW_WORDS + j;  // wave-uniform
      uint64_t bits = 0;
      if (word < nwords) {
        bits = cand[word];
        if (act && lane == 0) act[word] = bits;
        if (bits && lane == 0) cand[word] = 0ull;
      }
      int cls = -1;
      const uint64_t v = word * 64 + lane;
      if (bits && v < V && ((bits >> lane) & 1ull)) {
        const uint64_t len = ptr[v + 1] - ptr[v];
        if (len <= KC_SMALL) cls = 0;
        else if (len > KC_GIANT) cls = -1;
        // the block pass also takes the vertices whose answer may exceed the wave pass's bins
        else if (len > KC_HUGE || std::min<uint64_t>(len, est[v]) > KC_HIST) cls = 2;
        else cls = 1;
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        m[c][j] = __ballot(cls == c);
        n[c] += (uint32_t)__popcll(m[c][j]);
      }
    }
    if (!__syncthreads_or((int)(n[0] | n[1] | n[2]))) continue;
    if (lane == 0)
      for (int c = 0; c < 3; ++c) s_cnt[c][wave] = n[c];
    __syncthreads();
    if (threadIdx.x < 3) {
      uint32_t t = 0;
      for (int i = 0; i < 16; ++i) t += s_cnt[threadIdx.x][i];
      s_base[threadIdx.x] = t ? atomicAdd(threadIdx.x == 0 ? &cnt->nsmall : threadIdx.x == 1 ? &cnt->nbig : &cnt->nhuge,
                                          (unsigned long long)t)
                              : 0ull;
    }
    __syncthreads();
    if (n[0] | n[1] | n[2]) {
      uint64_t at[3];
      for (int c = 0; c < 3; ++c) {
        at[c] = s_base[c];
        for (int i = 0; i < wave; ++i) at[c] += s_cnt[c][i];
      }
#pragma unroll
      for (int j = 0; j < KC_CW_WORDS; ++j) {
        const uint32_t v = (uint32_t)((w0 + (uint64_t)wave * KC_CW_WORDS + j) * 64 + lane);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          if ((m[c][j] >> lane) & 1ull) {
            const uint64_t p = at[c] + (uint64_t)__popcll(m[c][j] & below);
            if (c == 0) qsmall[p] = v;
            else if (c == 1) qbig[p] = v;
            else *(qhuge_end - p) = v;  // the block pass's queue grows down from the end of qbig's array
          }
          at[c] += (uint64_t)__popcll(m[c][j]);
        }
      }
    }
    __syncthreads();  // s_cnt and s_base are rewritten by the next step
  }
}

// ---- h-index: lanes and waves -------------------------------------------------------------
// Largest i in [1, top] with (count of bins >= i) >= i from a wave's histogram (top <= KC_HIST;
// 0: none): lane l owns bins [PER l, PER l + PER), and the bins of the lanes above it are
// suffix-summed.  Every lane gets the answer.
__device__ __forceinline__ uint32_t kc_wave_pick(const uint32_t* hist, uint32_t top) {
  const int lane = threadIdx.x & 63;
  const uint32_t j0 = (uint32_t)lane * KC_PER;
  uint32_t own = 0;
  for (uint32_t j = j0; j < j0 + KC_PER && j <= top; ++j) own += hist[j];
  uint32_t incl = own;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_down(incl, off, 64);
    if (lane + off < 64) incl += t;
  }
  uint32_t best = 0, sum = incl - own;
  for (int j = (int)std::min(j0 + KC_PER - 1, top); j >= (int)j0 && j >= 1; --j) {
    sum += hist[j];
    if (sum >= (uint32_t)j) {
      best = (uint32_t)j;
      break;
    }
  }
  for (int off = 32; off > 0; off >>= 1) best = std::max(best, (uint32_t)__shfl_xor(best, off, 64));
  return best;
}

// the same from one lane's byte histogram
__device__ __forceinline__ uint32_t kc_lane_pick(const uint8_t* h, uint32_t top) {
  uint32_t sum = 0;
  for (uint32_t j = top; j > 0; --j) {
    sum += h[j];
    if (sum >= j) return j;
  }
  return 0;
}

__device__ __forceinline__ void kc_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The wave pass's vertices first (the longer ones), then one lane per vertex of the small
// queue.  A wave's LDS share serves both: KC_PER words per lane as one histogram of the
// wave, or KC_SMALL + 1 bytes per lane.  cnt_v: the counts, with the answers that the last spread
// found already (KC_AHEAD), nullptr without counts.
__global__ __launch_bounds__(KC_THREADS) void k_kc_hindex(
    const uint32_t* __restrict__ qsmall, const uint32_t* __restrict__ qbig, const kc_counters* __restrict__ cnt_in,
    const uint64_t* __restrict__ ptr, const uint32_t* __restrict__ idx, const uint32_t* __restrict__ est,
    const uint32_t* __restrict__ cnt_v, uint32_t* __restrict__ core) {
  __shared__ uint32_t hist_all[KC_THREADS / 64][64 * KC_PER];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t* hist = hist_all[wave];
  const uint64_t nbig = cnt_in->nbig, nsmall = cnt_in->nsmall;
  const uint64_t wave_id = grid_wave_id(), nwaves = grid_waves();
  for (uint64_t q = wave_id; q < nbig; q += nwaves) {
    const uint32_t v = qbig[q];
    const uint32_t known = cnt_v ? cnt_v[v] : 0u;
    if (known & KC_AHEAD) {  // uniform
      if (lane == 0) core[v] = known & ~KC_AHEAD;
      continue;
    }
    const uint64_t b = ptr[v], e = ptr[v + 1];
    const uint32_t top = (uint32_t)std::min<uint64_t>(e - b, (uint64_t)est[v]);  // at most KC_HIST
    for (uint32_t j = lane; j <= top; j += 64) hist[j] = 0;
    kc_wave_fence();
    for (uint64_t k0 = b; k0 < e; k0 += 64 * KC_U) {
      uint32_t eu[KC_U];
#pragma unroll
      for (int i = 0; i < KC_U; ++i) {
        const uint64_t k = k0 + (uint64_t)i * 64 + lane;
        eu[i] = k < e ? est[idx[k]] : 0u;
      }
#pragma unroll
      for (int i = 0; i < KC_U; ++i)
        if (k0 + (uint64_t)i * 64 + lane < e) atomicAdd(&hist[eu[i] < top ? eu[i] : top], 1u);
    }
    kc_wave_fence();
    const uint32_t best = kc_wave_pick(hist, top);
    if (lane == 0 && best && best < core[v]) core[v] = best;
    kc_wave_fence();
  }
  uint8_t* h = reinterpret_cast<uint8_t*>(hist) + lane * (KC_SMALL + 1);
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < nsmall;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t v = qsmall[i];
    const uint32_t known = cnt_v ? cnt_v[v] : 0u;
    if (known & KC_AHEAD) {
      core[v] = known & ~KC_AHEAD;
      continue;
    }
    const uint64_t b = ptr[v], e = ptr[v + 1];
    if (b == e) {
      core[v] = 0;  // kcore.hpp:214-218
      continue;
    }
    const uint32_t cap = std::min<uint32_t>((uint32_t)(e - b), est[v]);
    for (uint32_t j = 0; j <= cap; ++j) h[j] = 0;
    for (uint64_t k = b; k < e; ++k) {
      const uint32_t eu = est[idx[k]];
      ++h[eu < cap ? eu : cap];
    }
    const uint32_t best = kc_lane_pick(h, cap);
    if (best && best < core[v]) core[v] = best;
  }
}

// ---- h-index: blocks -------------------------------------------------------------------------
// shift of the first round over values up to cap: cap >> shift fits the bins
__device__ __forceinline__ int kc_first_shift(uint32_t cap) {
  int s = 0;
  while ((cap >> s) > KC_HHIST) ++s;
  return s;
}

// One round over bins hist[0..nb] of width 2^shift that start at base, with `above`
// neighbours over them: J = the largest j with above + (bins >= j) >= base + (j << shift)
// (j = 0 always holds) and the count over bin J.  Every thread calls it.
__device__ void kc_block_pick(const uint32_t* hist, uint32_t nb, uint32_t base, int shift, uint32_t above,
                              uint32_t* J, uint32_t* over) {
  __shared__ uint32_t s_wave[KC_HTHREADS / 64];
  __shared__ uint32_t s_best, s_over;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int WAVES = KC_HTHREADS / 64;
  // thread t owns bins [17 t, 17 t + 17); suffix sums over the threads above it
  const uint32_t j0 = (uint32_t)tid * KC_HPER;
  uint32_t own = 0;
  for (uint32_t j = j0; j < j0 + KC_HPER && j <= nb; ++j) own += hist[j];
  uint32_t incl = own;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_down(incl, off, 64);
    if (lane + off < 64) incl += t;
  }
  if (lane == 0) s_wave[wave] = incl;  // the wave's total
  if (tid == 0) {
    s_best = 0;
    s_over = 0;
  }
  __syncthreads();
  uint32_t sum = above + incl - own;
  for (int w = wave + 1; w < WAVES; ++w) sum += s_wave[w];
  uint32_t best = 0, mine = 0;
  bool has = false;
  for (int64_t j = (int64_t)std::min(j0 + KC_HPER - 1, nb); j >= (int64_t)j0; --j) {
    const uint32_t o = sum;
    sum += hist[j];
    if (j == 0 || sum >= base + ((uint32_t)j << shift)) {
      best = (uint32_t)j;
      mine = o;
      has = true;
      break;
    }
  }
  uint32_t wbest = best;
  for (int off = 32; off > 0; off >>= 1) wbest = std::max(wbest, (uint32_t)__shfl_xor(wbest, off, 64));
  if (lane == 0 && wbest) atomicMax(&s_best, wbest);
  __syncthreads();
  if (has && best == s_best) s_over = mine;  // one thread owns bin J
  __syncthreads();
  *J = s_best;
  *over = s_over;
  __syncthreads();  // the shared words are free again
}

// One block per queued vertex of up to KC_GIANT neighbours.
__global__ __launch_bounds__(KC_HTHREADS) void k_kc_huge(
    const uint32_t* __restrict__ qhuge_end, const kc_counters* __restrict__ cnt_in, const uint64_t* __restrict__ ptr,
    const uint32_t* __restrict__ idx, const uint32_t* __restrict__ est,
    const uint32_t* __restrict__ cnt_v, uint32_t* __restrict__ core) {
  __shared__ uint32_t hist[KC_HTHREADS * KC_HPER];
  const int tid = threadIdx.x;
  const uint64_t nhuge = cnt_in->nhuge;
  for (uint64_t q = blockIdx.x; q < nhuge; q += gridDim.x) {
    const uint32_t v = *(qhuge_end - q);
    const uint32_t known = cnt_v ? cnt_v[v] : 0u;
    if (known & KC_AHEAD) {  // uniform
      if (tid == 0) core[v] = known & ~KC_AHEAD;
      continue;
    }
    const uint64_t b = ptr[v], e = ptr[v + 1];
    const uint32_t cap = (uint32_t)std::min<uint64_t>(e - b, (uint64_t)est[v]);
    int shift = kc_first_shift(cap);
    uint32_t base = 0, above = 0, nb = cap >> shift;
    for (;;) {  // two rounds at most: cap < 2^28
      for (uint32_t j = tid; j <= nb; j += KC_HTHREADS) hist[j] = 0;
      __syncthreads();
      for (uint64_t k0 = b; k0 < e; k0 += KC_HTHREADS * KC_U) {
        uint32_t eu[KC_U];
#pragma unroll
        for (int i = 0; i < KC_U; ++i) {
          const uint64_t k = k0 + (uint64_t)i * KC_HTHREADS + tid;
          eu[i] = k < e ? est[idx[k]] : 0u;
        }
#pragma unroll
        for (int i = 0; i < KC_U; ++i) {
          const uint32_t x = std::min(eu[i], cap);
          const uint32_t j = (x - base) >> shift;
          if (k0 + (uint64_t)i * KC_HTHREADS + tid < e && x >= base && j <= nb) atomicAdd(&hist[j], 1u);
        }
      }
      __syncthreads();
      uint32_t J, over;
      kc_block_pick(hist, nb, base, shift, above, &J, &over);
      base += J << shift;
      above = over;
      if (shift == 0) break;
      const int ns = std::max(0, shift - (int)KC_HBITS);
      nb = (1u << (shift - ns)) - 1u;
      shift = ns;
    }
    if (tid == 0 && base && base < core[v]) core[v] = base;
  }
}

// Giants (more than KC_GIANT neighbours): their adjacencies in chunks of KC_GCHUNK, one
// block per chunk, each adding its LDS histogram of the neighbours' capped estimates into
// the giant's histogram in global memory (ghist, KC_HHIST + 1 bins per giant, zero between
// launches); then one block per giant picks from it.  Answers above KC_HHIST take another
// round.  Only giants with their bit in `act` are counted.
__global__ __launch_bounds__(KC_HTHREADS) void k_kc_giant_hist(
    const uint64_t* __restrict__ ptr, const uint32_t* __restrict__ idx, const uint32_t* __restrict__ giants,
    const unsigned long long* __restrict__ ngiant, const uint64_t* __restrict__ start,
    const uint64_t* __restrict__ act, const uint32_t* __restrict__ est, const kc_giant* __restrict__ state, int round,
    uint32_t* __restrict__ ghist) {
  __shared__ uint32_t hist[KC_HHIST + 1];
  const int tid = threadIdx.x;
  const uint64_t n = *ngiant;
  if (n == 0) return;
  const uint64_t total = start[n];
  for (uint64_t c = blockIdx.x; c < total; c += gridDim.x) {
    uint64_t k0, k1, gi;
    const uint32_t v = hub_chunk(ptr, giants, start, n, KC_GCHUNK, c, &k0, &k1, &gi);
    if (!((act[v >> 6] >> (v & 63)) & 1ull)) continue;  // uniform
    const uint32_t cap = (uint32_t)std::min<uint64_t>(ptr[v + 1] - ptr[v], (uint64_t)est[v]);
    int shift = kc_first_shift(cap);
    uint32_t base = 0, nb = cap >> shift;
    if (round) {
      const kc_giant g = state[gi];
      if (g.shift < 0) continue;  // uniform
      base = g.base;
      shift = g.shift;
      nb = g.nb;
    }
    for (uint32_t j = tid; j <= nb; j += KC_HTHREADS) hist[j] = 0;
    __syncthreads();
    for (uint64_t kk = k0; kk < k1; kk += KC_HTHREADS * KC_U) {
      uint32_t eu[KC_U];
#pragma unroll
      for (int i = 0; i < KC_U; ++i) {
        const uint64_t k = kk + (uint64_t)i * KC_HTHREADS + tid;
        eu[i] = k < k1 ? est[idx[k]] : 0u;
      }
#pragma unroll
      for (int i = 0; i < KC_U; ++i) {
        const uint32_t x = std::min(eu[i], cap);
        const uint32_t j = (x - base) >> shift;
        if (kk + (uint64_t)i * KC_HTHREADS + tid < k1 && x >= base && j <= nb) atomicAdd(&hist[j], 1u);
      }
    }
    __syncthreads();
    uint32_t* gh = ghist + gi * (uint64_t)(KC_HHIST + 1);
    for (uint32_t j = tid; j <= nb; j += KC_HTHREADS)
      if (hist[j]) atomicAdd(&gh[j], hist[j]);
    __syncthreads();
  }
}

__global__ __launch_bounds__(KC_HTHREADS) void k_kc_giant_pick(
    const uint64_t* __restrict__ ptr, const uint32_t* __restrict__ giants,
    const unsigned long long* __restrict__ ngiant, const uint64_t* __restrict__ act,
    const uint32_t* __restrict__ est, kc_giant* __restrict__ state, int round, uint32_t* __restrict__ ghist,
    uint32_t* __restrict__ core, uint32_t* __restrict__ cnt_v, kc_counters* __restrict__ cnt) {
  __shared__ uint32_t hist[KC_HTHREADS * KC_HPER];
  const int tid = threadIdx.x;
  const uint64_t n = *ngiant;
  for (uint64_t gi = blockIdx.x; gi < n; gi += gridDim.x) {
    const uint32_t v = giants[gi];
    if (!((act[v >> 6] >> (v & 63)) & 1ull)) continue;  // uniform
    const uint32_t cap = (uint32_t)std::min<uint64_t>(ptr[v + 1] - ptr[v], (uint64_t)est[v]);
    const int shift0 = kc_first_shift(cap);
    kc_giant g{0u, 0u, cap >> shift0, shift0};
    if (round) {
      g = state[gi];
      if (g.shift < 0) continue;  // uniform
    }
    uint32_t* gh = ghist + gi * (uint64_t)(KC_HHIST + 1);
    for (uint32_t j = tid; j <= g.nb; j += KC_HTHREADS) {
      hist[j] = gh[j];
      gh[j] = 0u;
    }
    __syncthreads();
    uint32_t J, over;
    kc_block_pick(hist, g.nb, g.base, g.shift, g.above, &J, &over);
    if (tid == 0) {
      g.base += J << g.shift;
      g.above = over;
      if (g.shift == 0) {
        g.shift = -1;
        if (g.base && g.base < core[v]) {
          core[v] = g.base;
          if (cnt_v) cnt_v[v] = 0u;  // re-counted chunk by chunk in the spread
        }
        atomicMax(&cnt->giant_top, (unsigned long long)core[v]);
      } else {
        const int ns = std::max(0, g.shift - (int)KC_HBITS);
        g.nb = (1u << (g.shift - ns)) - 1u;
        g.shift = ns;
      }
      state[gi] = g;
    }
    __syncthreads();
  }
}

// ---- spread ------------------------------------------------------------------------------------
// The modified vertices (core below est) activate their neighbours; with counts (cnt_v) each
// also takes itself out of the counts of the unmodified neighbours it fell below, marking those
// that the last one leaves short as candidates, and returns how many neighbours it keeps at or
// above its own new value.  The next active set is marked with plain stores that any number of
// waves may repeat, where an atomic OR on a shared bitmap word is serialized in the memory-side
// atomic unit (RMAT scale 22, all epochs: 35 ms of spreading with bits, 10 ms with bytes).  The
// mark is the top bit of the neighbour's coreness, which stands still meanwhile, so a
// neighbour costs one random read, where values of 31 bits suffice (act_bytes is nullptr then:
// with counts, and below 2^31 entries, so no length needs the bit; the lane and wave spreads 5.4 -> 4.2 ms, the
// blocks' 4.5 -> 4.8); else one byte per vertex.
static constexpr uint32_t KC_MARK = 0x80000000u;
struct kc_spread {
  const uint32_t* idx;
  const uint32_t* est;
  uint32_t* core;
  uint32_t* cnt_v;
  uint8_t* act_bytes;
  uint64_t* cand;
  __device__ __forceinline__ uint32_t value(uint32_t raw) const { return act_bytes ? raw : raw & ~KC_MARK; }
  __device__ __forceinline__ uint32_t one(uint32_t u, uint32_t raw, uint32_t old, uint32_t now) const {
    if (act_bytes) {
      if (!act_bytes[u]) act_bytes[u] = 1;
    } else if (!(raw & KC_MARK)) {
      core[u] = raw | KC_MARK;
    }
    if (!cnt_v) return 0u;
    const uint32_t cu = value(raw);
    if (cu > now && cu <= old && est[u] == cu && atomicSub(&cnt_v[u], 1u) == cu) kc_set_bit(cand, u);
    return cu >= now ? 1u : 0u;
  }
  // entries b + i0, b + i0 + step, ... below e
  __device__ __forceinline__ uint32_t range(uint64_t b, uint64_t e, uint32_t i0, uint32_t step, uint32_t old,
                                            uint32_t now) const {
    uint32_t c = 0;
    for (uint64_t k0 = b; k0 < e; k0 += (uint64_t)step * KC_U) {
      uint32_t u[KC_U], cu[KC_U];
#pragma unroll
      for (int i = 0; i < KC_U; ++i) {
        const uint64_t k = k0 + (uint64_t)i * step + i0;
        u[i] = k < e ? idx[k] : 0u;
        cu[i] = k < e && cnt_v ? core[u[i]] : 0u;
      }
#pragma unroll
      for (int i = 0; i < KC_U; ++i)
        if (k0 + (uint64_t)i * step + i0 < e) c += one(u[i], cu[i], old, now);
    }
    return c;
  }
  // with counts: the same, and the capped new values into hist[0..now]
  __device__ __forceinline__ void range_hist(uint64_t b, uint64_t e, uint32_t i0, uint32_t step, uint32_t old,
                                             uint32_t now, uint32_t* hist) const {
    for (uint64_t k0 = b; k0 < e; k0 += (uint64_t)step * KC_U) {
      uint32_t u[KC_U], cu[KC_U];
#pragma unroll
      for (int i = 0; i < KC_U; ++i) {
        const uint64_t k = k0 + (uint64_t)i * step + i0;
        u[i] = k < e ? idx[k] : 0u;
        cu[i] = k < e ? core[u[i]] : 0u;
      }
#pragma unroll
      for (int i = 0; i < KC_U; ++i)
        if (k0 + (uint64_t)i * step + i0 < e) {
          (void)one(u[i], cu[i], old, now);
          const uint32_t x = value(cu[i]);
          atomicAdd(&hist[x < now ? x : now], 1u);
        }
    }
  }
  // one lane's list
  __device__ __forceinline__ void range_lane(uint64_t b, uint64_t e, uint32_t old, uint32_t now, uint8_t* h) const {
    for (uint64_t k0 = b; k0 < e; k0 += KC_U) {
      uint32_t u[KC_U], cu[KC_U];
#pragma unroll
      for (int i = 0; i < KC_U; ++i) {
        u[i] = k0 + i < e ? idx[k0 + i] : 0u;
        cu[i] = k0 + i < e ? core[u[i]] : 0u;
      }
#pragma unroll
      for (int i = 0; i < KC_U; ++i)
        if (k0 + i < e) {
          (void)one(u[i], cu[i], old, now);
          const uint32_t x = value(cu[i]);
          ++h[x < now ? x : now];
        }
    }
  }
};

// With counts a spread's walk also takes the histogram of the neighbours' new values, capped at
// the vertex's own: it holds both its count and, when that falls short, its h-index of the next
// epoch, whose estimates are these values.  The vertex is then a candidate of the next epoch
// for sure, drops there, and counts anew, so its count's place carries the answer there
// (KC_AHEAD) and saves a second walk (RMAT scale 22, all
// epochs: h-index passes 7.0 -> 3.0 ms, spreads 10.2 -> 10.5 ms).  A block's vertex with a value above
// KC_HHIST and a giant have too many values for that and are walked again.
__global__ __launch_bounds__(KC_THREADS) void k_kc_spread(
    const uint32_t* __restrict__ qsmall, const uint32_t* __restrict__ qbig, const kc_counters* __restrict__ cnt_in,
    const uint64_t* __restrict__ ptr, kc_spread sp) {
  __shared__ uint32_t hist_all[KC_THREADS / 64][64 * KC_PER];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t* hist = hist_all[wave];
  const uint64_t nbig = cnt_in->nbig, nsmall = cnt_in->nsmall;
  const uint64_t wave_id = grid_wave_id(), nwaves = grid_waves();
  for (uint64_t q = wave_id; q < nbig; q += nwaves) {
    const uint32_t v = qbig[q];
    const uint32_t old = sp.est[v], now = sp.value(sp.core[v]);
    if (old == now) continue;  // uniform
    if (!sp.cnt_v) {
      (void)sp.range(ptr[v], ptr[v + 1], (uint32_t)lane, 64u, old, now);
      continue;
    }
    for (uint32_t j = lane; j <= now; j += 64) hist[j] = 0;
    kc_wave_fence();
    sp.range_hist(ptr[v], ptr[v + 1], (uint32_t)lane, 64u, old, now, hist);
    kc_wave_fence();
    const uint32_t c = hist[now];
    const uint32_t best = c < now ? kc_wave_pick(hist, now) : 0u;
    if (lane == 0) sp.cnt_v[v] = best ? best | KC_AHEAD : c;
    kc_wave_fence();
  }
  uint8_t* h = reinterpret_cast<uint8_t*>(hist) + lane * (KC_SMALL + 1);
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < nsmall;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t v = qsmall[i];
    const uint32_t old = sp.est[v], now = sp.value(sp.core[v]);
    if (old == now) continue;
    if (!sp.cnt_v || old == KC_UNSET) {
      (void)sp.range(ptr[v], ptr[v + 1], 0u, 1u, old, now);
      continue;
    }
    for (uint32_t j = 0; j <= now; ++j) h[j] = 0;
    sp.range_lane(ptr[v], ptr[v + 1], old, now, h);
    const uint32_t c = h[now];
    const uint32_t best = c < now ? kc_lane_pick(h, now) : 0u;
    sp.cnt_v[v] = best ? best | KC_AHEAD : c;
  }
}

__global__ __launch_bounds__(KC_HTHREADS) void k_kc_spread_huge(const uint32_t* __restrict__ qhuge_end,
                                                                const kc_counters* __restrict__ cnt_in,
                                                                const uint64_t* __restrict__ ptr, kc_spread sp) {
  __shared__ uint32_t hist[KC_HTHREADS * KC_HPER];
  __shared__ uint32_t s_c;
  const uint32_t tid = threadIdx.x;
  const uint64_t nhuge = cnt_in->nhuge;
  for (uint64_t q = blockIdx.x; q < nhuge; q += gridDim.x) {
    const uint32_t v = *(qhuge_end - q);
    const uint32_t old = sp.est[v], now = sp.value(sp.core[v]);
    if (old == now) continue;  // uniform
    if (!sp.cnt_v) {
      (void)sp.range(ptr[v], ptr[v + 1], tid, KC_HTHREADS, old, now);
      continue;
    }
    if (now <= KC_HHIST) {  // uniform
      for (uint32_t j = tid; j <= now; j += KC_HTHREADS) hist[j] = 0;
      __syncthreads();
      sp.range_hist(ptr[v], ptr[v + 1], tid, KC_HTHREADS, old, now, hist);
      __syncthreads();
      const uint32_t c = hist[now];
      uint32_t best = 0, over;
      if (c < now) kc_block_pick(hist, now, 0u, 0, 0u, &best, &over);
      if (tid == 0) sp.cnt_v[v] = best ? best | KC_AHEAD : c;
    } else {
      if (tid == 0) s_c = 0u;
      __syncthreads();
      uint32_t c = sp.range(ptr[v], ptr[v + 1], tid, KC_HTHREADS, old, now);
      for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
      if ((tid & 63) == 0) atomicAdd(&s_c, c);
      __syncthreads();
      if (tid == 0) sp.cnt_v[v] = s_c;
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(KC_HTHREADS) void k_kc_spread_giant(const uint64_t* __restrict__ ptr,
                                                                 const uint32_t* __restrict__ giants,
                                                                 const unsigned long long* __restrict__ ngiant,
                                                                 const uint64_t* __restrict__ start,
                                                                 const uint64_t* __restrict__ act, kc_spread sp) {
  const uint64_t n = *ngiant;
  if (n == 0) return;
  const uint64_t total = start[n];
  for (uint64_t c = blockIdx.x; c < total; c += gridDim.x) {
    uint64_t k0, k1;
    const uint32_t v = hub_chunk(ptr, giants, start, n, KC_GCHUNK, c, &k0, &k1);
    if (!((act[v >> 6] >> (v & 63)) & 1ull)) continue;  // uniform
    const uint32_t old = sp.est[v], now = sp.value(sp.core[v]);
    if (old == now) continue;
    uint32_t k = sp.range(k0, k1, threadIdx.x, KC_HTHREADS, old, now);
    if (sp.cnt_v) {
      for (int off = 32; off > 0; off >>= 1) k += __shfl_xor(k, off, 64);
      if ((threadIdx.x & 63) == 0 && k) atomicAdd(&sp.cnt_v[v], k);
    }
  }
}

// ---- commit --------------------------------------------------------------------------------------
// estimate = coreness for the epoch's candidates (kcore.hpp:248-258); modified ones that are
// already short again stay candidates.
__global__ __launch_bounds__(KC_THREADS) void k_kc_commit(
    const uint32_t* __restrict__ qsmall, const uint32_t* __restrict__ qbig, const uint32_t* __restrict__ qhuge_end,
    const uint32_t* __restrict__ giants, const unsigned long long* __restrict__ ngiant,
    const uint64_t* __restrict__ act, const uint32_t* __restrict__ core, uint32_t mark, uint32_t* __restrict__ est,
    const uint32_t* __restrict__ cnt_v, uint64_t* __restrict__ cand, kc_counters* __restrict__ cnt) {
  const uint64_t ns = cnt->nsmall, nb = cnt->nbig, nh = cnt->nhuge, ng = giants ? *ngiant : 0ull;
  unsigned long long nmod = 0;
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < ns + nb + nh + ng;
       i += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t v;
    if (i < ns) {
      v = qsmall[i];
    } else if (i < ns + nb) {
      v = qbig[i - ns];
    } else if (i < ns + nb + nh) {
      v = *(qhuge_end - (i - ns - nb));
    } else {
      v = giants[i - ns - nb - nh];
      if (!((act[v >> 6] >> (v & 63)) & 1ull)) continue;
    }
    const uint32_t c = core[v] & ~mark, old = est[v];
    if (c == old) continue;
    est[v] = c;
    nmod += old != KC_UNSET ? 1u : 0u;
    if (cnt_v) {
      const uint32_t n = cnt_v[v];
      if (n < c || (n & KC_AHEAD)) kc_set_bit(cand, v);
    }
  }
  block_add2(nmod, 0, &cnt->modified, &cnt->modified);
}

// sizes of the next active set (its bytes, cleared here) and candidate set; without counts the
// active set is the candidate set
__global__ __launch_bounds__(256) void k_kc_next(uint64_t* __restrict__ act_bytes, uint64_t* __restrict__ cand,
                                                 uint64_t nwords, int is_cand, kc_counters* __restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  const uint64_t n = nwords * 8;  // 8-byte groups of marks; eight lanes cover one bitmap word
  unsigned long long a = 0, c = 0;
  for (uint64_t base = grid_wave_id() * 64; base < n; base += grid_waves() * 64) {
    const uint64_t i = base + lane;
    uint64_t w = 0;
    if (i < n) {
      w = act_bytes[i];
      if (w) act_bytes[i] = 0ull;
    }
    a += (unsigned long long)__popcll(w);
    if (is_cand) {
      uint64_t bits = ((w * 0x0102040810204080ull) >> 56) << ((lane & 7) * 8);  // byte j's mark -> bit j
      for (int off = 4; off > 0; off >>= 1) bits |= __shfl_xor(bits, off, 64);
      if (i < n && (lane & 7) == 0) cand[i >> 3] = bits;
    } else if (i < n && (lane & 7) == 0) {
      c += (unsigned long long)__popcll(cand[i >> 3]);
    }
  }
  if (is_cand) c = a;
  block_add2(a, c, &cnt->next_active, &cnt->next_cand);
}

// the same where the marks are top bits of the values
__global__ __launch_bounds__(1024) void k_kc_next_marked(uint32_t* __restrict__ core, uint64_t V,
                                                         const uint64_t* __restrict__ cand, uint64_t nwords,
                                                         kc_counters* __restrict__ cnt) {
  const uint64_t i0 = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, step = (uint64_t)gridDim.x * blockDim.x;
  unsigned long long a = 0, c = 0;
  uint4* quads = reinterpret_cast<uint4*>(core);
  for (uint64_t i = i0; i < V / 4; i += step) {
    const uint4 x = quads[i];
    const uint32_t n = (x.x >> 31) + (x.y >> 31) + (x.z >> 31) + (x.w >> 31);
    if (n) quads[i] = make_uint4(x.x & ~KC_MARK, x.y & ~KC_MARK, x.z & ~KC_MARK, x.w & ~KC_MARK);
    a += n;
  }
  if (i0 < V % 4) {
    const uint64_t v = V - V % 4 + i0;
    const uint32_t x = core[v];
    a += x >> 31;
    core[v] = x & ~KC_MARK;
  }
  for (uint64_t i = i0; i < nwords; i += step) c += (unsigned long long)__popcll(cand[i]);
  block_add2(a, c, &cnt->next_active, &cnt->next_cand);
}

}  // namespace pe

using namespace pe;

// byte_marks_from: adjacency entries from which on the active marks are bytes (see kc_spread);
// the values have 31 bits below 2^31 entries
static constexpr uint64_t KC_MARKED_BELOW = 1ull << 31;

static int kcore_run(pe_graph_t* g, int out_edges, uint64_t byte_marks_from, uint32_t* coreness,
                     uint64_t* epoch_modified, uint64_t* epoch_next, uint32_t cap, pe_kcore_stats_t* stats) {
  if (!g || !coreness) return PE_ERR_INVALID;
  return guarded(g->ctx, [&] {
    PE_REQUIRE(!out_edges || g->has_csr, PE_ERR_STATE, "out-edge k-core needs PE_GRAPH_BUILD_CSR");
    pe_ctx_s* ctx = g->ctx;
    hipStream_t s = ctx->stream;
    const uint32_t V = g->V;
    const uint64_t* ptr = out_edges ? g->csr_ptr() : g->col_ptr.p;
    const uint32_t* idx = out_edges ? g->csr_idx() : g->row_idx.p;
    const bool counts = g->csr_is_csc;  // the adjacency is its own reverse
    const uint64_t nwords = ((uint64_t)V >> 6) + 1;
    const uint32_t Vs = std::max<uint32_t>(1, V);
    dbuf<uint32_t> core(ctx, Vs), est(ctx, Vs), qsmall(ctx, Vs), cnt_v;
    // the other queues: every vertex in them holds more than KC_SMALL of the entries
    const uint64_t nlong = std::min<uint64_t>(Vs, g->nnz / (KC_SMALL + 1) + 1);
    dbuf<uint32_t> qbig(ctx, nlong);
    // active marks in the values' top bits
    const bool marked = counts && g->nnz < std::min(byte_marks_from, KC_MARKED_BELOW);
    dbuf<uint64_t> cand(ctx, nwords), act, nxt;             // nxt: else, one byte per vertex
    if (!marked) nxt.alloc(ctx, nwords * 8);
    if (counts) cnt_v.alloc(ctx, Vs);
    uint32_t* qhuge_end = qbig.p + (nlong - 1);
    dbuf<kc_counters> cnt(ctx, 2);  // two sets: consecutive epochs alternate
    PE_HIP(hipEventRecord(ctx->t0, s));
    k_kc_init<<<grid_for(V, 256, 8192), 256, 0, s>>>(ptr, V, core.p, est.p, cnt_v.p);
    k_kc_fill<<<grid_for(nwords, 256, 4096), 256, 0, s>>>(cand.p, nwords, V);  // active_current.fill()
    if (!marked) k_kc_zero<<<grid_for(nwords * 8, 256, 4096), 256, 0, s>>>(nxt.p, nwords * 8);
    PE_HIP(hipGetLastError());
    // giants and their histograms (one per giant, KC_HHIST + 1 bins)
    hub_table giants;
    hub_table_build(ctx, ptr, V, g->nnz, KC_GIANT, KC_GCHUNK, giants);
    const uint64_t ngiant = mail_post(ctx, giants.count.p, 1, reinterpret_cast<unsigned long long*>(cnt.p), 2 * KC_CW)[0];
    const uint64_t ghist_words = ngiant * (uint64_t)(KC_HHIST + 1);
    dbuf<uint32_t> ghist;
    dbuf<kc_giant> gstate;
    if (ngiant) {
      act.alloc(ctx, nwords);
      ghist.alloc(ctx, ghist_words + 1);  // whole 8-byte words to clear
      gstate.alloc(ctx, ngiant);
      k_kc_zero<<<grid_for((ghist_words + 1) / 2, 256, 4096), 256, 0, s>>>(reinterpret_cast<uint64_t*>(ghist.p),
                                                                          (ghist_words + 1) / 2);
      PE_HIP(hipGetLastError());
    }
    const kc_spread sp{idx, est.p, core.p, cnt_v.p, reinterpret_cast<uint8_t*>(nxt.p), cand.p};
    const unsigned full_grid = persistent_grid(ctx, 1u << 20, 8), huge_max = persistent_grid(ctx, 1u << 20, 2);
    const uint32_t* gl = ngiant ? giants.hubs.p : nullptr;
    uint32_t epoch = 0;
    uint64_t total_mod = 0, ncand = V, giant_top = g->nnz;
    for (;;) {
      kc_counters* c = cnt.p + (epoch & 1);
      uint64_t modified = 0, next = 0;
      if (ncand) {
        const unsigned grid = (unsigned)std::min<uint64_t>(full_grid, (ncand + 3) / 4);
        const unsigned hgrid = (unsigned)std::min<uint64_t>(huge_max, ncand);
        k_kc_classify<<<grid_for(nwords, 16 * KC_CW_WORDS, (unsigned)std::max(1, ctx->num_cus) * 2), 1024, 0, s>>>(
            cand.p, act.p, nwords, V, ptr, est.p, qsmall.p, qbig.p, qhuge_end, c);
        k_kc_huge<<<hgrid, KC_HTHREADS, 0, s>>>(qhuge_end, c, ptr, idx, est.p, cnt_v.p, core.p);
        k_kc_hindex<<<grid, KC_THREADS, 0, s>>>(qsmall.p, qbig.p, c, ptr, idx, est.p, cnt_v.p, core.p);
        if (ngiant) {
          // rounds: 14 bits of the answer each after the first
          int rounds = 1;
          for (uint64_t t = std::min<uint64_t>(giant_top, 0xFFFFFFFEull); t > KC_HHIST; t >>= KC_HBITS) ++rounds;
          const unsigned pgrid = (unsigned)std::min<uint64_t>(ngiant, huge_max);
          for (int r = 0; r < rounds; ++r) {
            k_kc_giant_hist<<<huge_max, KC_HTHREADS, 0, s>>>(ptr, idx, gl, giants.count.p, giants.start.p, act.p, est.p,
                                                             gstate.p, r, ghist.p);
            k_kc_giant_pick<<<pgrid, KC_HTHREADS, 0, s>>>(ptr, gl, giants.count.p, act.p, est.p, gstate.p, r, ghist.p,
                                                          core.p, cnt_v.p, c);
          }
          k_kc_spread_giant<<<huge_max, KC_HTHREADS, 0, s>>>(ptr, gl, giants.count.p, giants.start.p, act.p, sp);
        }
        k_kc_spread_huge<<<hgrid, KC_HTHREADS, 0, s>>>(qhuge_end, c, ptr, sp);
        k_kc_spread<<<grid, KC_THREADS, 0, s>>>(qsmall.p, qbig.p, c, ptr, sp);
        k_kc_commit<<<grid_for(ncand, KC_THREADS, full_grid), KC_THREADS, 0, s>>>(
            qsmall.p, qbig.p, qhuge_end, gl, giants.count.p, act.p, core.p, marked ? KC_MARK : 0u, est.p, cnt_v.p, cand.p, c);
        const unsigned next_max = (unsigned)std::max(1, ctx->num_cus) * 2;
        if (marked) k_kc_next_marked<<<grid_for(V, 4096, next_max), 1024, 0, s>>>(core.p, V, cand.p, nwords, c);
        else k_kc_next<<<grid_for(nwords * 8, 256, next_max), 256, 0, s>>>(nxt.p, cand.p, nwords, counts ? 0 : 1, c);
        PE_HIP(hipGetLastError());
        const kc_counters* h = reinterpret_cast<const kc_counters*>(
            mail_post(ctx, reinterpret_cast<const unsigned long long*>(c), KC_CW,
                      reinterpret_cast<unsigned long long*>(cnt.p + ((epoch + 1) & 1)), KC_CW));
        modified = h->modified;
        next = h->next_active;
        ncand = h->next_cand;
        if (epoch == 0) giant_top = h->giant_top;  // estimates only fall from here on
      }
      if (epoch < cap && epoch_modified) epoch_modified[epoch] = modified;
      if (epoch < cap && epoch_next) epoch_next[epoch] = next;  // need_modified
      total_mod += modified;
      ++epoch;
      if (next == 0) break;  // kcore.hpp:264
      // every epoch but the last lowers some coreness, which starts at most at its length
      PE_REQUIRE((uint64_t)epoch <= g->nnz + 2, PE_ERR_INTERNAL, "k-core did not terminate");
    }
    PE_HIP(hipEventRecord(ctx->t1, s));
    PE_HIP(hipEventSynchronize(ctx->t1));
    float ms = 0.f;
    PE_HIP(hipEventElapsedTime(&ms, ctx->t0, ctx->t1));
    download_external(g, core.p, coreness, 4);
    if (stats) {
      stats->epochs = epoch;
      stats->modified = total_mod;
      stats->seconds = ms * 1e-3;
    }
  });
}

extern "C" int pe_kcore(pe_graph_t* g, int out_edges, uint32_t* coreness, uint64_t* epoch_modified,
                        uint64_t* epoch_next, uint32_t cap, pe_kcore_stats_t* stats) {
  return kcore_run(g, out_edges, KC_MARKED_BELOW, coreness, epoch_modified, epoch_next, cap, stats);
}

extern "C" int pe_kcore_byte_marks(pe_graph_t* g, int out_edges, uint64_t byte_marks_from, uint32_t* coreness,
                                   uint64_t* epoch_modified, uint64_t* epoch_next, uint32_t cap,
                                   pe_kcore_stats_t* stats) {
  return kcore_run(g, out_edges, byte_marks_from, coreness, epoch_modified, epoch_next, cap, stats);
}
