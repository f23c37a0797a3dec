// HyperANF: plato::algo::hyperanf (plato/algo/hyperanf/hyperanf.hpp:80-197) on the device.
//
// Every vertex holds a HyperLogLog counter of 2^P one-byte registers
// (plato/util/hyperloglog.hpp:32-142), started with its own id (MurmurHash3_x86_32 of
// the 4-byte id, seed 0x5f61767a: register = hash >> (32 - P), rank = 1 + leading
// zeros of hash << P, at most 33 - P).  An iteration gives every vertex the
// register-wise max of its counter and its in-neighbours' counters of the previous
// iteration: the reference's push (active vertices merge into their out-neighbours'
// deltas) and pull (every vertex merges its in-neighbours) deliver exactly that, since
// a counter that did not change was already merged downstream.  Register max is
// order-independent, so the counters are bit-exact; anf is the FP64 sum of the
// per-vertex estimates, and the loop stops after `iterations` or when anf grows by less
// than DBL_EPSILON (that anf is dropped).  The average distance is GetAvgDistance over
// the anfs (hyperanf.hpp:58-67).
//
// Layout: counters [V][2^P] bytes, double-buffered (Jacobi), read as 16 registers per lane
// and load: LPR = 2^P / 16 lanes hold a row (at most 64; counters above 1024 registers walk
// the in-edges once per 1024), so a wave's load brings 64 / LPR rows.  A row that the last
// iteration left as it was has already been merged by its out-neighbours, so a bitmap of the
// changed rows decides per in-edge whether the row is read at all, a vertex without changed
// in-neighbours is not touched, and its estimate is kept.  No row of a vertex that someone
// pulls from can pass the register-wise max over the first counters of all such vertices (the
// bound row): a pull stops at the first row that reaches it, and a vertex that has reached it
// is done.  The pull's bound is the random 2^P-byte rows of the second and third iteration,
// then the in-edge lists.  RMAT scale 23 symmetrized, P = 6, 8 pulls: 5.2 ms each with one
// 4-byte word per lane and every row read; here 1.8, 3.4 and 2.5 ms, then 0.8 falling to 0.15 ms
// (without the bound row 3.4 until the fourth, then 0.8); the whole call 44.7 -> 13.4 ms.
// Three passes by in-degree: fewer than HANF_LOW_DEG, a group of LPR lanes per vertex; up to
// HANF_HUB_DEG, a wave per vertex; the hubs' in-edges in chunks over all waves, each merging
// its chunk's maximum into the hub's row, so no wave walks a hub alone.
#include <cfloat>
#include <cmath>
#include <vector>

#include "pe_internal.hpp"

namespace pe {

static constexpr uint64_t HANF_HUB_DEG = 4096;    // in-edges above which a vertex is a hub
static constexpr uint64_t HANF_HUB_CHUNK = 2048;  // in-edges of a hub per wave task
static constexpr uint64_t HANF_LOW_DEG = 32;    // fewer in-edges take a lane group per vertex
static constexpr int HANF_U = 8;                 // rows a lane keeps in flight at most

__device__ __forceinline__ uint32_t hanf_rotl(uint32_t x, int r) { return (x << r) | (x >> (32 - r)); }

// MurmurHash3_x86_32 of one little-endian 32-bit word (len 4), the reference's hash of
// a vertex id (plato/util/hash.hpp:33-96, A. Appleby's published algorithm)
__device__ __forceinline__ uint32_t hanf_murmur_u32(uint32_t key, uint32_t seed) {
  uint32_t k = key * 0xcc9e2d51u;
  k = hanf_rotl(k, 15);
  k *= 0x1b873593u;
  uint32_t h = seed ^ k;
  h = hanf_rotl(h, 13);
  h = h * 5 + 0xe6546b64u;
  h ^= 4u;
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

// register and rank of a vertex's own id
__device__ __forceinline__ void hanf_first(uint32_t id, int P, uint32_t* reg, uint32_t* rank) {
  const uint32_t h = hanf_murmur_u32(id, 0x5f61767au);
  const uint32_t w = h << P;
  const uint32_t q = 32u - (uint32_t)P;
  const uint32_t r = w ? (uint32_t)__clz(w) + 1u : q + 1u;
  *reg = h >> q;
  *rank = r < q + 1u ? r : q + 1u;
}

// Counters of at most 2^HANF_CODE_P registers start as a 16-bit code, register << 6 | rank:
// the first pull reads 2 bytes per in-edge instead of a row that holds one register.
static constexpr int HANF_CODE_P = 10;
__global__ void k_hanf_codes(uint16_t* __restrict__ code, uint32_t V, int P, const uint32_t* __restrict__ perm) {
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t reg, rank;
    hanf_first(perm ? perm[v] : (uint32_t)v, P, &reg, &rank);  // counters hash input ids
    code[v] = (uint16_t)(reg << 6 | rank);
  }
}

// the 16 registers from 16 w on of a row that starts as `code`
__device__ __forceinline__ uint4 hanf_code_row(uint32_t code, uint32_t w) {
  const uint32_t reg = code >> 6, at = (reg >> 4) == w ? (reg >> 2) & 3u : 4u;
  const uint32_t x = (code & 63u) << ((reg & 3u) * 8u);
  return make_uint4(at == 0 ? x : 0u, at == 1 ? x : 0u, at == 2 ? x : 0u, at == 3 ? x : 0u);
}

__global__ void k_hanf_init_rows(uint4* __restrict__ rows, uint32_t V, uint32_t log_wpr4,
                                 const uint16_t* __restrict__ code) {
  const uint64_t n = (uint64_t)V << log_wpr4, mask = (1ull << log_wpr4) - 1ull;
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    rows[i] = hanf_code_row(code[i >> log_wpr4], (uint32_t)(i & mask));
}

__global__ void k_hanf_init(uint8_t* __restrict__ regs, uint32_t V, int P, const uint32_t* __restrict__ perm) {
  const uint64_t m = 1ull << P;
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t reg, rank;
    hanf_first(perm ? perm[v] : (uint32_t)v, P, &reg, &rank);
    regs[v * m + reg] = (uint8_t)rank;
  }
}

__global__ void k_hanf_zero(uint32_t* __restrict__ p, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

// Byte-wise max of many words: the odd bytes in 16-bit maxima of the words as they are (the
// high byte decides, the low byte only breaks ties), the even bytes in those of the words
// shifted up by one byte: three instructions per word of four registers, where unpacking
// each byte takes about sixteen.
typedef uint16_t hanf_u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(hanf_u16x2, a),
                                                                __builtin_bit_cast(hanf_u16x2, b)));
}

__device__ __forceinline__ uint32_t byte_max4(uint32_t a, uint32_t b) {
  return (max_u16x2(a, b) & 0xFF00FF00u) | ((max_u16x2(a << 8, b << 8) >> 8) & 0x00FF00FFu);
}

struct row_max {  // 16 registers
  uint32_t odd[4] = {0, 0, 0, 0}, even[4] = {0, 0, 0, 0};
  __device__ __forceinline__ void add(const uint4& r) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      odd[i] = max_u16x2(odd[i], w[i]);
      even[i] = max_u16x2(even[i], w[i] << 8);
    }
  }
  __device__ __forceinline__ uint4 row() const {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (odd[i] & 0xFF00FF00u) | ((even[i] >> 8) & 0x00FF00FFu);
    return make_uint4(w[0], w[1], w[2], w[3]);
  }
};

__device__ __forceinline__ uint4 row_max2(const uint4& a, const uint4& b) {
  return make_uint4(byte_max4(a.x, b.x), byte_max4(a.y, b.y), byte_max4(a.z, b.z), byte_max4(a.w, b.w));
}
__device__ __forceinline__ uint4 row_shfl_xor(const uint4& a, int off) {
  return make_uint4((uint32_t)__shfl_xor((int)a.x, off, 64), (uint32_t)__shfl_xor((int)a.y, off, 64),
                    (uint32_t)__shfl_xor((int)a.z, off, 64), (uint32_t)__shfl_xor((int)a.w, off, 64));
}
__device__ __forceinline__ bool row_differs(const uint4& a, const uint4& b) {
  return ((a.x ^ b.x) | (a.y ^ b.y) | (a.z ^ b.z) | (a.w ^ b.w)) != 0u;
}

// the lanes g * LPR of the groups of LPR lanes that are all set in m
template <int LPR>
__device__ __forceinline__ uint64_t full_groups(uint64_t m) {
#pragma unroll
  for (int k = 1; k < LPR; k <<= 1) m &= m >> k;
  constexpr uint64_t first = LPR == 64 ? 1ull : ~0ull / ((1ull << (LPR & 63)) - 1ull);  // every LPR-th bit
  return m & first;
}

// The bound row: register-wise max of the first counters of the vertices with out-degree (od),
// or with entries in their own list (ptr), one word per register, zeroed before.  Registers
// that fit are collected per block in LDS.
static constexpr uint32_t HANF_LDS_REGS = 4096;
__global__ __launch_bounds__(256) void k_hanf_bound(uint32_t V, int P, const uint32_t* __restrict__ perm,
                                                    const uint32_t* __restrict__ od, const uint64_t* __restrict__ ptr,
                                                    uint32_t* __restrict__ top) {
  __shared__ uint32_t s_top[HANF_LDS_REGS];
  const uint32_t m = 1u << P;
  const bool lds = m <= HANF_LDS_REGS;
  if (lds) {
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) s_top[i] = 0u;
    __syncthreads();
  }
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
    if (od ? od[v] == 0u : ptr[v] == ptr[v + 1]) continue;
    uint32_t reg, rank;
    hanf_first(perm ? perm[v] : (uint32_t)v, P, &reg, &rank);
    uint32_t* t = lds ? &s_top[reg] : &top[reg];
    if (*t < rank) atomicMax(t, rank);
  }
  if (lds) {
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x)
      if (s_top[i] > top[i]) atomicMax(&top[i], s_top[i]);
  }
}

__global__ void k_hanf_bound_row(const uint32_t* __restrict__ top, uint32_t m, uint8_t* __restrict__ row) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) row[i] = (uint8_t)top[i];
}

__global__ void k_hanf_fill_bits(uint64_t* __restrict__ w, uint64_t nwords, uint32_t V) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < nwords; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t lo = i * 64;
    w[i] = lo + 64 <= V ? ~0ull : (lo < V ? (1ull << (V - lo)) - 1ull : 0ull);
  }
}

// vertices of the wave-per-vertex pass: lo <= in-degree <= HANF_HUB_DEG
__global__ __launch_bounds__(256) void k_hanf_mid_bits(const uint64_t* __restrict__ ptr, uint32_t V, uint64_t nwords,
                                                       uint64_t lo, uint64_t* __restrict__ bits) {
  const int lane = threadIdx.x & 63;
  for (uint64_t word = grid_wave_id(); word < nwords; word += grid_waves()) {
    const uint64_t v = word * 64 + lane;
    bool in = false;
    if (v < V) {
      const uint64_t d = ptr[v + 1] - ptr[v];
      in = d >= lo && d <= HANF_HUB_DEG;
    }
    const uint64_t m = __ballot(in);
    if (lane == 0) bits[word] = m;
  }
}

// One byte per vertex: bit 0, its row changed in the last pull; bit 1, it has reached the bound.
static constexpr uint8_t HANF_CHANGED = 1, HANF_DONE = 2;

// The changed marks as a bitmap, and whether there is any.
__global__ __launch_bounds__(256) void k_hanf_bits(const uint64_t* __restrict__ bytes, uint64_t nwords,
                                                   uint64_t* __restrict__ bits, unsigned long long* __restrict__ any) {
  const int lane = threadIdx.x & 63;
  const uint64_t n = nwords * 8;
  bool got = false;
  for (uint64_t base = grid_wave_id() * 64; base < n; base += grid_waves() * 64) {
    const uint64_t i = base + lane;
    const uint64_t w = i < n ? bytes[i] & 0x0101010101010101ull : 0ull;
    uint64_t b = ((w * 0x0102040810204080ull) >> 56) << ((lane & 7) * 8);  // byte j's mark -> bit j
    for (int off = 4; off > 0; off >>= 1) b |= __shfl_xor(b, off, 64);
    if (i < n && (lane & 7) == 0) bits[i >> 3] = b;
    got |= w != 0;
  }
  if (__ballot(got) && lane == 0) *any = 1ull;
}

// Max over the rows of the changed in-neighbours in [b, e) (words c0.. of each row), folded
// over the wave's 64 / LPR row slots: every lane gets its 16 registers.  Returns whether there
// was any.  The ids come 64 at a time, one per lane; the changed ones are packed to the front
// with one forward permute, so that every row load of the wave is full.  A slot that reaches
// the bound row's words (bound) ends the walk.
template <int LPR>
__device__ __forceinline__ bool hanf_range(uint64_t b, uint64_t e, const uint32_t* __restrict__ row_idx,
                                           const uint64_t* __restrict__ changed, const uint4* __restrict__ cur,
                                           uint64_t wpr4, uint64_t c0, const uint4& bound, uint4* out) {
  constexpr int S = 64 / LPR, U = S * HANF_U > 64 ? 64 / S : HANF_U;
  const int lane = threadIdx.x & 63, slot = lane / LPR, w = lane % LPR;
  const uint64_t below = (1ull << lane) - 1ull;
  row_max acc;
  bool any = false;
  for (uint64_t k0 = b; k0 < e; k0 += 64) {
    uint32_t u = 0;
    bool on = false;
    if (k0 + lane < e) {
      u = row_idx[k0 + lane];
      on = (changed[u >> 6] >> (u & 63)) & 1ull;
    }
    const uint64_t m = __ballot(on);
    const uint32_t n = (uint32_t)__popcll(m);
    if (n == 0) continue;
    any = true;
    const uint32_t to = on ? (uint32_t)__popcll(m & below) : n + (uint32_t)__popcll(~m & below);
    const uint32_t id = (uint32_t)__builtin_amdgcn_ds_permute((int)(to << 2), (int)u);
    for (uint32_t t = 0; t < n; t += S * U) {
      uint4 r[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const uint32_t k = t + (uint32_t)(i * S + slot);
        const uint32_t x = (uint32_t)__shfl((int)id, (int)(k & 63u), 64);
        r[i] = k < n ? cur[(uint64_t)x * wpr4 + c0 + w] : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < U; ++i) acc.add(r[i]);
    }
    if (full_groups<LPR>(__ballot(!row_differs(acc.row(), bound)))) break;
  }
  uint4 r = acc.row();
  if (any)
    for (int off = LPR; off < 64; off <<= 1) r = row_max2(r, row_shfl_xor(r, off));
  *out = r;
  return any;
}

// The same for the first pull, from the codes: one LDS maximum per in-edge into the wave's
// registers (s, one word each).  Making each row from its code in registers instead took
// 1.36 ms for the wave pass at RMAT scale 23, reading the rows 1.97 ms, this 0.91 ms (hubs 0.97,
// 0.62 and 0.51 ms).
template <int LPR>
__device__ __forceinline__ bool hanf_first_range(uint64_t b, uint64_t e, const uint32_t* __restrict__ row_idx,
                                                 const uint16_t* __restrict__ code, uint32_t* s, uint4* out) {
  constexpr uint32_t M = 16 * LPR;
  constexpr int U = 4;
  const uint32_t lane = threadIdx.x & 63, w = lane % LPR;
#pragma unroll
  for (uint32_t i = 0; i < M; i += 64) s[i + lane] = 0u;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  for (uint64_t k0 = b; k0 < e; k0 += 64 * U) {
    uint32_t c[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const uint64_t k = k0 + (uint64_t)i * 64 + lane;
      c[i] = k < e ? (uint32_t)code[row_idx[k]] : 0u;  // rank 0: no effect
    }
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (c[i]) atomicMax(&s[c[i] >> 6], c[i] & 63u);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  uint32_t r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t* q = s + w * 16 + i * 4;
    r[i] = q[0] | q[1] << 8 | q[2] << 16 | q[3] << 24;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();  // read before the wave's next vertex clears them
  *out = make_uint4(r[0], r[1], r[2], r[3]);
  return b < e;
}

// A vertex's row is written to the next buffer when it changes now, or when it changed last
// time (the next buffer then still holds the row before that).
template <int LPR, bool FIRST>
__global__ __launch_bounds__(256) void k_hanf_pull_wave(const uint64_t* __restrict__ col_ptr,
                                                        const uint32_t* __restrict__ row_idx,
                                                        const uint32_t* __restrict__ queue,
                                                        const unsigned long long* __restrict__ nq, uint64_t wpr4,
                                                        const uint64_t* __restrict__ changed,
                                                        const uint16_t* __restrict__ code,
                                                        const uint4* __restrict__ bound_row,
                                                        const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                                        uint8_t* __restrict__ marks) {
  __shared__ uint32_t s_regs[FIRST ? 4 : 1][FIRST ? 16 * LPR : 1];
  const int lane = threadIdx.x & 63, w = lane % LPR;
  const uint64_t n = *nq, nwaves = grid_waves();
  for (uint64_t q = grid_wave_id(); q < n; q += nwaves) {
    const uint32_t v = queue[q];
    const uint8_t was = marks[v];
    if (was == HANF_DONE) continue;  // done, and in both buffers
    const uint64_t b = col_ptr[v], e = (was & HANF_DONE) ? b : col_ptr[v + 1];
    const bool stale = (changed[v >> 6] >> (v & 63)) & 1ull;
    bool mark = false, done = true;
    for (uint64_t c0 = 0; c0 < wpr4; c0 += LPR) {
      const uint4 bound = bound_row[c0 + w];
      uint4 r;
      bool any;
      if constexpr (FIRST) any = hanf_first_range<LPR>(b, e, row_idx, code, s_regs[threadIdx.x >> 6], &r);
      else any = hanf_range<LPR>(b, e, row_idx, changed, cur, wpr4, c0, bound, &r);
      if (!any && !stale) {
        done = false;  // as it was: not done
        continue;
      }
      const uint64_t at = (uint64_t)v * wpr4 + c0 + w;
      const uint4 own = cur[at];
      const uint4 now = row_max2(own, r);
      const bool diff = __ballot(row_differs(own, now)) != 0ull;
      mark |= diff;
      done &= __ballot(row_differs(now, row_max2(now, bound))) == 0ull;
      if ((diff || stale) && lane < LPR) nxt[at] = now;
    }
    if (lane == 0) marks[v] = (uint8_t)((mark ? HANF_CHANGED : 0) | (done ? HANF_DONE : 0));
  }
}

// A group of LPR lanes per vertex of fewer than HANF_LOW_DEG in-edges, 64 / LPR vertices per
// wave step, LPR in-edges of each at a time (an id per lane), so that the vertices' short
// chains of dependent loads overlap.
template <int LPR, bool FIRST>
__global__ __launch_bounds__(256) void k_hanf_pull_low(const uint64_t* __restrict__ col_ptr,
                                                       const uint32_t* __restrict__ row_idx, uint32_t V,
                                                       const uint64_t* __restrict__ changed,
                                                       const uint16_t* __restrict__ code,
                                                       const uint4* __restrict__ bound_row,
                                                       const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                                       uint8_t* __restrict__ marks) {
  constexpr int G = 64 / LPR, U = LPR < HANF_U ? LPR : HANF_U;
  const int lane = threadIdx.x & 63, grp = lane / LPR, w = lane % LPR, g0 = grp * LPR;
  const uint64_t nwaves = grid_waves();
  const uint4 bound = bound_row[w];
  for (uint64_t v0 = grid_wave_id() * G; v0 < V; v0 += nwaves * G) {
    const uint64_t v = v0 + grp;
    uint64_t b = 0, e = 0;
    bool mine = false, stale = false;
    uint8_t was = 0;
    if (v < V) {
      was = marks[v];
      b = col_ptr[v];
      e = col_ptr[v + 1];
      mine = e - b < HANF_LOW_DEG && was != HANF_DONE;  // done, and in both buffers
      stale = (changed[v >> 6] >> (v & 63)) & 1ull;
    }
    if (!mine || (was & HANF_DONE)) e = b;
    row_max acc;
    bool any = false;
    for (uint64_t k0 = b; __ballot(k0 < e) != 0ull; k0 += LPR) {  // until the wave's longest list is done
      uint32_t u = 0;
      bool on = false;
      if (k0 + w < e) {
        u = row_idx[k0 + w];
        on = FIRST || ((changed[u >> 6] >> (u & 63)) & 1ull);
        if (FIRST) u = code[u];
      }
      const uint64_t m = (__ballot(on) >> g0) & (LPR == 64 ? ~0ull : (1ull << LPR) - 1ull);  // the group's
      any |= m != 0ull;
#pragma unroll
      for (int t = 0; t < LPR; t += U) {
        uint4 r[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const uint32_t x = (uint32_t)__shfl((int)u, g0 + t + i, 64);
          r[i] = !((m >> (t + i)) & 1ull) ? make_uint4(0, 0, 0, 0)
                 : FIRST                  ? hanf_code_row(x, (uint32_t)w)
                                          : cur[(uint64_t)x * LPR + w];
        }
#pragma unroll
        for (int i = 0; i < U; ++i) acc.add(r[i]);
      }
      const uint64_t full = full_groups<LPR>(__ballot(!row_differs(acc.row(), bound)));
      if ((full >> g0) & 1ull) e = b;  // at the bound: nothing left to gain
    }
    bool diff = false, below = true;
    if (mine && (any || stale)) {
      const uint4 own = cur[v * LPR + w];
      const uint4 now = row_max2(own, acc.row());
      diff = row_differs(own, now);
      below = row_differs(now, row_max2(now, bound));
      if (diff || stale) nxt[v * LPR + w] = now;
    }
    const uint64_t dm = (__ballot(diff) >> g0) & (LPR == 64 ? ~0ull : (1ull << LPR) - 1ull);
    // a lane whose own registers stay still writes them when others of the row change
    if (dm && !diff && !stale) nxt[v * LPR + w] = cur[v * LPR + w];
    const uint64_t bm = (__ballot(below) >> g0) & (LPR == 64 ? ~0ull : (1ull << LPR) - 1ull);
    if (mine && w == 0) marks[v] = (uint8_t)((dm ? HANF_CHANGED : 0) | (bm ? 0 : HANF_DONE));
  }
}

// The hubs' own rows, before their in-edges.
__global__ __launch_bounds__(256) void k_hanf_hub_rows(const uint32_t* __restrict__ hubs,
                                                       const unsigned long long* __restrict__ nhub, uint64_t wpr4,
                                                       const uint4* __restrict__ bound_row,
                                                       const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                                       uint8_t* __restrict__ marks) {
  const int lane = threadIdx.x & 63;
  const uint64_t n = *nhub, nwaves = grid_waves();
  for (uint64_t h = grid_wave_id(); h < n; h += nwaves) {
    const uint64_t v = hubs[h];
    bool below = false;
    for (uint64_t i = lane; i < wpr4; i += 64) {
      const uint4 own = cur[v * wpr4 + i];
      below |= row_differs(own, row_max2(own, bound_row[i]));
      nxt[v * wpr4 + i] = own;
    }
    const bool done = __ballot(below) == 0ull;
    if (lane == 0) marks[v] = done ? HANF_DONE : 0;
  }
}

// Register-wise max of x into *p (a compare-and-swap loop: every retry sees a word that
// only grew, so it ends); whether *p grew.
__device__ __forceinline__ bool byte_max_merge(uint32_t* p, uint32_t x) {
  uint32_t old = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    const uint32_t nv = byte_max4(old, x);
    if (nv == old) return false;
    const uint32_t prev = atomicCAS(p, old, nv);
    if (prev == old) return true;
    old = prev;
  }
}

// Hub in-edges, one chunk per wave at a time, the chunk's max merged into the hub's next row.
template <int LPR, bool FIRST>
__global__ __launch_bounds__(256) void k_hanf_pull_hubs(const uint64_t* __restrict__ col_ptr,
                                                        const uint32_t* __restrict__ row_idx,
                                                        const uint32_t* __restrict__ hubs,
                                                        const unsigned long long* __restrict__ nhub,
                                                        const uint64_t* __restrict__ start, uint64_t wpr4,
                                                        const uint64_t* __restrict__ changed,
                                                        const uint16_t* __restrict__ code,
                                                        const uint4* __restrict__ bound_row,
                                                        const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                                        uint8_t* __restrict__ marks) {
  __shared__ uint32_t s_regs[FIRST ? 4 : 1][FIRST ? 16 * LPR : 1];
  const int lane = threadIdx.x & 63;
  const uint64_t nwaves = grid_waves();
  const uint64_t n = *nhub;
  if (n == 0) return;
  const uint64_t total = start[n];
  for (uint64_t c = grid_wave_id(); c < total; c += nwaves) {
    uint64_t k0, k1;
    const uint32_t v = hub_chunk(col_ptr, hubs, start, n, HANF_HUB_CHUNK, c, &k0, &k1);
    if (marks[v] & HANF_DONE) continue;  // uniform
    for (uint64_t c0 = 0; c0 < wpr4; c0 += LPR) {
      uint4 r;
      if constexpr (FIRST) (void)hanf_first_range<LPR>(k0, k1, row_idx, code, s_regs[threadIdx.x >> 6], &r);
      else if (!hanf_range<LPR>(k0, k1, row_idx, changed, cur, wpr4, c0, bound_row[c0 + lane % LPR], &r)) continue;
      if (lane < LPR) {
        uint32_t* p = reinterpret_cast<uint32_t*>(nxt + (uint64_t)v * wpr4 + c0 + lane);
        const bool grew = byte_max_merge(p, r.x) | byte_max_merge(p + 1, r.y) | byte_max_merge(p + 2, r.z) |
                          byte_max_merge(p + 3, r.w);
        if (grew) marks[v] = HANF_CHANGED;
      }
    }
  }
}

// 2^-r exactly, from the exponent bits (r <= 33)
__device__ __forceinline__ double hanf_pow2_neg(uint32_t r) {
  return __longlong_as_double((long long)(1023u - r) << 52);
}

// The estimate of one counter from its register sum s (exact: at most 2^16 terms of 2^-r)
// and its zero registers (hyperloglog.hpp:77-116, with its small- and large-range
// corrections); alpha is alpha_m * m^2.
__device__ __forceinline__ double hanf_estimate(double alpha, double m, double s, uint32_t zeros) {
  double est = alpha / s;
  if (est <= 5.0 / 2.0 * m) {
    if (zeros) est = m * log(m / zeros);
  } else if (est > (1.0 / 30.0) * 4294967296.0) {
    est = -4294967296.0 * log(1.0 - (est / 4294967296.0));
  }
  return est;
}

__device__ __forceinline__ double hanf_alpha(int P) {
  const double m = (double)(1u << P);
  double alpha;
  switch (P) {
    case 4: alpha = 0.673; break;
    case 5: alpha = 0.697; break;
    case 6: alpha = 0.709; break;
    default: alpha = 0.7213 / (1.0 + 1.079 / m); break;
  }
  return alpha * m * m;
}

// Estimates of counters of at most 1024 registers, summed per block in a fixed order:
// m / 16 lanes per counter (16 registers each, one 16-byte load), 1024 / m counters per
// wave step, so a wave keeps many counters' loads in flight instead of one.  Only changed
// counters are read; the others' estimates are kept in est (nullptr: every counter is read).
// Without `changed` every counter is a first one: one register set, whose rank the small-range
// estimate does not use.
__global__ __launch_bounds__(256) void k_hanf_estimate_rows(const uint8_t* __restrict__ regs, uint32_t V, int P,
                                                            const uint64_t* __restrict__ changed,
                                                            double* __restrict__ est, double* __restrict__ part) {
  __shared__ double s_w[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t m = 1u << P, L = m / 16, sub = (uint32_t)lane % L, slot = (uint32_t)lane / L, per = 64 / L;
  const double alpha = hanf_alpha(P);
  const uint64_t wave_id = grid_wave_id(), nwaves = grid_waves();
  double total = 0.0;  // lane's running sum over its counters, in order
  for (uint64_t v0 = wave_id * per; v0 < V; v0 += nwaves * per) {
    const uint64_t v = v0 + slot;
    double s = 0.0;
    uint32_t zeros = 0;
    const bool on = v < V && (!changed || !est || ((changed[v >> 6] >> (v & 63)) & 1ull));
    if (!changed) {
      s = sub == 0 ? (double)m : 0.0;
      zeros = sub == 0 ? m - 1u : 0u;
    } else if (on) {
      const uint4 q = *reinterpret_cast<const uint4*>(regs + v * m + (uint64_t)sub * 16);
      const uint32_t w4[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int b = 0; b < 32; b += 8) {
          const uint32_t r = (w4[i] >> b) & 0xFFu;
          s += hanf_pow2_neg(r);
          zeros += r == 0 ? 1u : 0u;
        }
    }
    for (uint32_t off = 1; off < L; off <<= 1) {
      s += __shfl_xor(s, (int)off, 64);
      zeros += (uint32_t)__shfl_xor((int)zeros, (int)off, 64);
    }
    if (v < V && sub == 0) {
      const double x = on ? hanf_estimate(alpha, (double)m, s, zeros) : est[v];
      if (on && est) est[v] = x;
      total += x;
    }
  }
  for (int off = 32; off > 0; off >>= 1) total += __shfl_down(total, off, 64);
  if (lane == 0) s_w[wave] = total;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Per-vertex estimate (hyperloglog.hpp:77-116) of larger counters, one wave per counter,
// summed per block in a fixed order.
// The register sum of 2^-reg is exact in FP64 (at most 2^16 terms of 2^-k, k <= 27).
__global__ __launch_bounds__(256) void k_hanf_estimate(const uint8_t* __restrict__ regs, uint32_t V, int P,
                                                       const uint64_t* __restrict__ changed,
                                                       double* __restrict__ est, double* __restrict__ part) {
  __shared__ double s_w[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t m = 1ull << P;
  const uint64_t wave_id = grid_wave_id(), nwaves = grid_waves();
  const double alpha = hanf_alpha(P);
  double total = 0.0;  // lane 0's running sum over this wave's vertices, in order
  for (uint64_t v = wave_id; v < V; v += nwaves) {
    if (changed && est && !((changed[v >> 6] >> (v & 63)) & 1ull)) {  // uniform
      total += est[v];
      continue;
    }
    double s = 0.0;
    uint32_t zeros = 0;
    for (uint64_t i = lane; i < m; i += 64) {
      const uint32_t r = regs[v * m + i];
      s += hanf_pow2_neg(r);
      zeros += r == 0 ? 1u : 0u;
    }
    for (int off = 32; off > 0; off >>= 1) {
      s += __shfl_xor(s, off, 64);
      zeros += __shfl_xor(zeros, off, 64);
    }
    const double x = hanf_estimate(alpha, (double)m, s, zeros);
    if (lane == 0 && est) est[v] = x;
    total += x;
  }
  if (lane == 0) s_w[wave] = total;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// n-step degrees: the estimate of each target's counter as the reference stores it,
// static_cast<vid_t>(estimate) - 1 (nstepdegrees.hpp:412-421); 0 for other vertices.
// One wave per vertex; targets (input ids, a bitmap) are looked up through perm.
__global__ __launch_bounds__(256) void k_nstep_degree(const uint8_t* __restrict__ regs, uint32_t V, int P,
                                                      const uint64_t* __restrict__ targets,
                                                      const uint32_t* __restrict__ perm, uint32_t* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const uint64_t m = 1ull << P;
  const uint64_t wave_id = grid_wave_id(), nwaves = grid_waves();
  const double alpha = hanf_alpha(P);
  for (uint64_t v = wave_id; v < V; v += nwaves) {
    const uint32_t id = perm ? perm[v] : (uint32_t)v;
    if (targets && !((targets[id >> 6] >> (id & 63)) & 1ull)) {
      if (lane == 0) out[v] = 0u;
      continue;
    }
    double s = 0.0;
    uint32_t zeros = 0;
    for (uint64_t i = lane; i < m; i += 64) {
      const uint32_t r = regs[v * m + i];
      s += hanf_pow2_neg(r);
      zeros += r == 0 ? 1u : 0u;
    }
    for (int off = 32; off > 0; off >>= 1) {
      s += __shfl_xor(s, off, 64);
      zeros += __shfl_xor(zeros, off, 64);
    }
    if (lane == 0) out[v] = (uint32_t)hanf_estimate(alpha, (double)m, s, zeros) - 1u;
  }
}

// counters in input-id order
__global__ void k_hanf_rows_external(const uint8_t* __restrict__ in, const uint32_t* __restrict__ rank_of,
                                     uint32_t V, uint64_t m, uint8_t* __restrict__ out) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < (uint64_t)V * m;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t v = i / m, j = i % m;
    out[i] = in[(uint64_t)rank_of[v] * m + j];
  }
}

}  // namespace pe

using namespace pe;

// An array that makes a call faster but that it can do without: empty when memory is short.
template <typename T>
static void hanf_alloc_optional(dbuf<T>& b, pe_ctx_s* ctx, size_t n) {
  try {
    b.alloc(ctx, n);
  } catch (const error& e) {
    if (e.code != PE_ERR_OOM) throw;
    b = dbuf<T>();
  }
}

// The pull over one adjacency (ptr, idx): its passes' vertex lists and the changed rows.
struct hanf_pull {
  pe_ctx_s* ctx;
  const uint64_t* ptr;
  const uint32_t* idx;
  uint32_t V;
  int P;
  uint64_t nwords;
  hub_table hubs;
  dbuf<uint32_t> mid;             // vertices of the wave pass
  dbuf<unsigned long long> nmid;  // [0] their number, [1] whether the last pull changed a row
  dbuf<uint64_t> changed;         // rows that the last pull changed (all before the first)
  dbuf<uint64_t> marks;           // HANF_CHANGED and HANF_DONE bytes
  dbuf<uint32_t> top;             // the bound row, a word per register
  dbuf<uint8_t> bound;            // the bound row
  dbuf<uint16_t> code;            // first counters, P <= HANF_CODE_P (empty when memory is short)
  bool first = true;              // no pull yet
  unsigned grid;

  // vertices of the wave pass at most: below 10 bits each has HANF_LOW_DEG of the entries
  static uint64_t max_mid(uint32_t V, uint64_t nnz, int bits) {
    const uint64_t Vs = std::max<uint32_t>(1, V);
    return bits < 10 ? std::min(Vs, nnz / HANF_LOW_DEG + 1) : Vs;
  }

  // od (out-degrees over this adjacency's entries) or, without it, src_ptr tells which vertices
  // some other vertex pulls from: those with od > 0, or with entries in src_ptr
  hanf_pull(pe_ctx_s* c, const uint64_t* p, const uint32_t* i, uint32_t v, uint64_t nnz, int bits, const uint32_t* perm,
            const uint32_t* od, const uint64_t* src_ptr)
      : ctx(c), ptr(p), idx(i), V(v), P(bits), nwords(((uint64_t)v >> 6) + 1), mid(c, max_mid(v, nnz, bits)),
        nmid(c, 2), changed(c, nwords), marks(c, nwords * 8), top(c, 1ull << bits), bound(c, 1ull << bits) {
    hipStream_t s = ctx->stream;
    k_hanf_zero<<<64, 256, 0, s>>>(top.p, 1ull << P);
    k_hanf_bound<<<persistent_grid(ctx, grid_for(V, 256), 4), 256, 0, s>>>(V, P, perm, od, src_ptr, top.p);
    k_hanf_bound_row<<<64, 256, 0, s>>>(top.p, 1u << P, bound.p);
    hub_table_build(ctx, ptr, V, nnz, HANF_HUB_DEG, HANF_HUB_CHUNK, hubs);
    // rows of 64 lanes and more have no group pass: the wave pass takes every shorter list
    k_hanf_zero<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t*>(nmid.p), 4);
    k_hanf_mid_bits<<<grid_for(nwords, 4, 8192), 256, 0, s>>>(ptr, V, nwords, P < 10 ? HANF_LOW_DEG : 0, changed.p);
    frontier_compact(ctx, changed.p, nwords, V, mid.p, nmid.p);
    k_hanf_fill_bits<<<grid_for(nwords, 256, 4096), 256, 0, s>>>(changed.p, nwords, V);
    k_hanf_zero<<<grid_for(nwords * 16, 256, 8192), 256, 0, s>>>(reinterpret_cast<uint32_t*>(marks.p), nwords * 16);
    if (P <= HANF_CODE_P) {
      hanf_alloc_optional(code, ctx, std::max<uint32_t>(1, V));
    }
    if (code.p) {
      k_hanf_codes<<<grid_for(V, 256, 8192), 256, 0, s>>>(code.p, V, P, perm);
    }
    PE_HIP(hipGetLastError());
    grid = persistent_grid(ctx, grid_for(V, 4), 8);
  }

  // the first counters
  void init(uint8_t* regs, uint64_t bytes, const uint32_t* perm) {
    hipStream_t s = ctx->stream;
    if (code.p) {
      k_hanf_init_rows<<<grid_for((uint64_t)V << (P - 4), 256, 65536), 256, 0, s>>>(reinterpret_cast<uint4*>(regs), V,
                                                                                   (uint32_t)P - 4u, code.p);
    } else {
      k_hanf_zero<<<grid_for(bytes / 4, 256, 65536), 256, 0, s>>>(reinterpret_cast<uint32_t*>(regs), bytes / 4);
      k_hanf_init<<<grid_for(V, 256, 8192), 256, 0, s>>>(regs, V, P, perm);
    }
    PE_HIP(hipGetLastError());
  }

  template <int LPR, bool FIRST>
  void launch(const uint4* cur, uint4* nxt) {
    hipStream_t s = ctx->stream;
    const uint64_t wpr4 = (1ull << P) / 16;
    uint8_t* mk = reinterpret_cast<uint8_t*>(marks.p);
    const uint4* br = reinterpret_cast<const uint4*>(bound.p);
    if constexpr (LPR < 64)
      k_hanf_pull_low<LPR, FIRST><<<grid, 256, 0, s>>>(ptr, idx, V, changed.p, code.p, br, cur, nxt, mk);
    k_hanf_pull_wave<LPR, FIRST><<<grid, 256, 0, s>>>(ptr, idx, mid.p, nmid.p, wpr4, changed.p, code.p, br, cur, nxt, mk);
    k_hanf_hub_rows<<<grid_for(hubs.max_hubs, 4, 1024), 256, 0, s>>>(hubs.hubs.p, hubs.count.p, wpr4, br, cur, nxt, mk);
    k_hanf_pull_hubs<LPR, FIRST><<<grid, 256, 0, s>>>(ptr, idx, hubs.hubs.p, hubs.count.p, hubs.start.p, wpr4, changed.p,
                                                      code.p, br, cur, nxt, mk);
  }

  // cur: the first counters before the first pull.  nxt[v] = register-wise max of cur[v] and cur[u] over the adjacency of v; nxt holds the
  // rows before the last pull (anything before the first)
  void pull(const uint8_t* cur, uint8_t* nxt) {
    const uint4* c = reinterpret_cast<const uint4*>(cur);
    uint4* n = reinterpret_cast<uint4*>(nxt);
    const bool from_codes = first && code.p;
    first = false;
    switch (P) {
      case 6: from_codes ? launch<4, true>(c, n) : launch<4, false>(c, n); break;
      case 7: from_codes ? launch<8, true>(c, n) : launch<8, false>(c, n); break;
      case 8: from_codes ? launch<16, true>(c, n) : launch<16, false>(c, n); break;
      case 9: from_codes ? launch<32, true>(c, n) : launch<32, false>(c, n); break;
      default: from_codes ? launch<64, true>(c, n) : launch<64, false>(c, n);
    }
    hipStream_t s = ctx->stream;
    k_hanf_zero<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t*>(nmid.p + 1), 2);
    k_hanf_bits<<<grid_for(nwords * 8, 256, 1024), 256, 0, s>>>(marks.p, nwords, changed.p, nmid.p + 1);
    PE_HIP(hipGetLastError());
  }
};

extern "C" int pe_hyperanf(pe_graph_t* g, const pe_hyperanf_opts_t* opts, double* anfs, uint32_t cap,
                           uint32_t* nanfs, double* avg_distance, uint8_t* registers, double* seconds) {
  if (!g || !opts || !anfs || cap == 0) return PE_ERR_INVALID;
  return guarded(g->ctx, [&] {
    const int P = (int)opts->bits;
    PE_REQUIRE(P >= 6 && P <= 16, PE_ERR_INVALID, "bits must be in [6, 16] (hyperanf_test supported range)");
    pe_ctx_s* ctx = g->ctx;
    hipStream_t s = ctx->stream;
    const uint32_t V = g->V;
    const uint64_t m = 1ull << P, bytes = std::max<uint64_t>(4, (uint64_t)V * m);
    dbuf<uint8_t> a(ctx, bytes), b(ctx, bytes);
    const unsigned est_grid = persistent_grid(ctx, grid_for(V, 4), 4);
    dbuf<double> part(ctx, est_grid);
    std::vector<double> hpart(est_grid);
    const uint32_t* perm = g->relabeled ? g->perm.p : nullptr;
    PE_HIP(hipEventRecord(ctx->t0, s));
    hanf_pull pulls(ctx, g->col_ptr.p, g->row_idx.p, V, g->nnz, P, perm, g->od.p, nullptr);
    dbuf<double> est;
    hanf_alloc_optional(est, ctx, std::max<uint32_t>(1, V));
    auto anf_of = [&](const uint8_t* regs) {
      const uint64_t* changed = pulls.first ? nullptr : pulls.changed.p;
      if (P <= 10)
        k_hanf_estimate_rows<<<est_grid, 256, 0, s>>>(regs, V, P, changed, est.p, part.p);
      else
        k_hanf_estimate<<<est_grid, 256, 0, s>>>(regs, V, P, changed, est.p, part.p);
      PE_HIP(hipGetLastError());
      PE_HIP(hipMemcpyAsync(hpart.data(), part.p, est_grid * sizeof(double), hipMemcpyDeviceToHost, s));
      PE_HIP(hipStreamSynchronize(s));
      double t = 0.0;
      for (double x : hpart) t += x;
      return t;
    };
    pulls.init(a.p, bytes, perm);
    std::vector<double> out;
    double last = anf_of(a.p);
    out.push_back(last);
    uint8_t* cur = a.p;
    uint8_t* nxt = b.p;
    for (uint32_t it = 0; it < opts->iterations; ++it) {
      pulls.pull(cur, nxt);
      const double anf = anf_of(nxt);
      std::swap(cur, nxt);
      if (anf - last < DBL_EPSILON) break;  // hyperanf.hpp:189-191
      out.push_back(anf);
      last = anf;
    }
    PE_HIP(hipEventRecord(ctx->t1, s));
    PE_HIP(hipEventSynchronize(ctx->t1));
    float ms = 0.f;
    PE_HIP(hipEventElapsedTime(&ms, ctx->t0, ctx->t1));
    for (size_t i = 0; i < out.size() && i < cap; ++i) anfs[i] = out[i];
    if (nanfs) *nanfs = (uint32_t)out.size();
    if (avg_distance) {  // GetAvgDistance (hyperanf.hpp:58-67)
      double avg = 0.0;
      for (size_t i = 1; i < out.size(); ++i) avg += i * (out[i] - out[i - 1]);
      *avg_distance = avg / (out.back() - out.front());
    }
    if (registers) {
      if (g->relabeled) {
        k_hanf_rows_external<<<grid_for((uint64_t)V * m, 256, 65536), 256, 0, s>>>(cur, g->rank_of.p, V, m, nxt);
        PE_HIP(hipGetLastError());
        host_download(ctx, nxt, registers, (uint64_t)V * m);
      } else {
        host_download(ctx, cur, registers, (uint64_t)V * m);
      }
    }
    if (seconds) *seconds = ms * 1e-3;
  });
}

extern "C" int pe_nstep_degrees(pe_graph_t* g, const uint64_t* target_words, uint32_t step, uint32_t bits,
                                int type, uint32_t* in_degrees, uint32_t* out_degrees, double* seconds) {
  if (!g) return PE_ERR_INVALID;
  return guarded(g->ctx, [&] {
    const int P = (int)bits;
    PE_REQUIRE(P >= 6 && P <= 16, PE_ERR_INVALID, "bits must be in [6, 16] (nstepdegrees supported range)");
    PE_REQUIRE(type >= PE_NSTEP_IN && type <= PE_NSTEP_BOTH, PE_ERR_INVALID, "type must be PE_NSTEP_IN, OUT or BOTH");
    PE_REQUIRE(!(type & PE_NSTEP_IN) || in_degrees, PE_ERR_INVALID, "in_degrees is required for the in pass");
    PE_REQUIRE(!(type & PE_NSTEP_OUT) || out_degrees, PE_ERR_INVALID, "out_degrees is required for the out pass");
    pe_ctx_s* ctx = g->ctx;
    hipStream_t s = ctx->stream;
    const uint32_t V = g->V;
    const uint64_t m = 1ull << P, bytes = std::max<uint64_t>(4, (uint64_t)V * m);
    const uint32_t* perm = g->relabeled ? g->perm.p : nullptr;
    dbuf<uint64_t> tw;
    if (target_words) {
      const uint64_t nw = ((uint64_t)V >> 6) + 1;
      tw.alloc(ctx, nw);
      PE_HIP(hipMemcpyAsync(tw.p, target_words, nw * 8, hipMemcpyHostToDevice, s));
    }
    dbuf<uint8_t> a(ctx, bytes), b(ctx, bytes);
    dbuf<uint32_t> dev_deg(ctx, std::max<uint32_t>(1, V));
    const unsigned grid = persistent_grid(ctx, grid_for(V, 4), 8);
    PE_HIP(hipEventRecord(ctx->t0, s));
    // one pass per direction: the in pass gathers over in-edges (the reference's
    // propagate on the forward engine), the out pass over out-edges (on the reversed one)
    auto pass = [&](const uint64_t* ptr, const uint32_t* idx, const uint32_t* od, const uint64_t* src_ptr,
                    uint32_t* host_out) {
      hanf_pull pulls(ctx, ptr, idx, V, g->nnz, P, perm, od, src_ptr);
      pulls.init(a.p, bytes, perm);
      uint8_t* cur = a.p;
      uint8_t* nxt = b.p;
      for (uint32_t it = 0; it < step; ++it) {  // nstepdegrees.hpp:343-409
        pulls.pull(cur, nxt);
        unsigned long long changed = 0;
        PE_HIP(hipMemcpyAsync(&changed, pulls.nmid.p + 1, 8, hipMemcpyDeviceToHost, s));
        PE_HIP(hipStreamSynchronize(s));
        std::swap(cur, nxt);
        if (!changed) break;  // no book grew: further steps change nothing
      }
      k_nstep_degree<<<grid, 256, 0, s>>>(cur, V, P, tw.p, perm, dev_deg.p);
      PE_HIP(hipGetLastError());
      download_external(g, dev_deg.p, host_out, 4);
    };
    if (type & PE_NSTEP_IN) pass(g->col_ptr.p, g->row_idx.p, g->od.p, nullptr, in_degrees);
    if (type & PE_NSTEP_OUT) {
      if (!g->directed && (type & PE_NSTEP_IN)) {
        std::memcpy(out_degrees, in_degrees, (size_t)V * 4);  // undirected: out = in (nstepdegrees.hpp:456-463)
      } else {
        PE_REQUIRE(g->has_csr || g->csr_is_csc, PE_ERR_STATE, "the out pass needs out-edges (PE_GRAPH_BUILD_CSR)");
        pass(g->csr_ptr(), g->csr_idx(), nullptr, g->col_ptr.p, out_degrees);
      }
    }
    PE_HIP(hipEventRecord(ctx->t1, s));
    PE_HIP(hipEventSynchronize(ctx->t1));
    float ms = 0.f;
    PE_HIP(hipEventElapsedTime(&ms, ctx->t0, ctx->t1));
    if (seconds) *seconds = ms * 1e-3;
  });
}
