// Connected components: plato::algo::connected_component_t::compute
// (plato/algo/cgm/connected_component.hpp:170-234) on the device engine.
//
// Labels start at the vertex ids and only ever take a smaller label: pushed along the
// out-edges of the vertices whose label changed in the last epoch (the push slot's
// write_min and set_bit, :193-205), or pulled by every vertex as the minimum of its
// own id and its in-neighbours' labels (:206-224).  The engine's rule picks push or
// pull per epoch from the active set's out-degree sum (dualmode.hpp:264-279), and the
// loop ends after an epoch that lowers no label.  The fixed point is unique: label(v)
// is the smallest input id from which v is reachable (on an undirected graph, the
// smallest id of its component), whatever the order in which labels spread; only the
// per-epoch activity depends on it, as in the reference, whose threads race the same way.
//
// Labels are kept in input ids, so a degree-relabeled graph gives the same labels.
//
// No label falls below the smallest id that has an out-edge (the floor): a pull stops at the
// first in-neighbour that carries it, and a vertex that has it is left alone.  A pull epoch
// takes the hubs first, then the vertices of more than CC_PULL_CAP in-edges, then the others,
// each pass reading what the ones before it wrote, so in a graph with one big component most
// vertices meet the floor's label at the head of their list in epoch 0 already.  RMAT scale 23
// symmetrized, degree-relabeled: 5.4 ms of pull epochs (1.8 ms each, all lists read to their
// ends, small ones first) against 0.8 and 0.1 ms; the whole call, whose components were
// counted on the host, 22.0 -> 5.9 ms, and 2.3 ms with the labels downloaded through pinned slots
// and the work arrays kept between calls.  Bound now by the labels' way to the host.
#include <algorithm>
#include <vector>

#include "pe_internal.hpp"

namespace pe {

static constexpr uint32_t CC_PULL_CAP = 64;  // in-edges a pull lane takes; longer go one wave each
static constexpr uint64_t CC_HUB_DEG = 4096;    // longer still: chunks of CC_HUB_CHUNK over all waves
static constexpr uint64_t CC_HUB_CHUNK = 2048;
static constexpr int CC_U = 4;                  // in-edges a lane loads per round trip

struct cc_counters {
  unsigned long long activated;     // sum of the slots' returns
  unsigned long long active_edges;  // out-edges of the next active set
  unsigned long long queued;        // push frontier size
  unsigned long long heavy;         // vertices of the wave-per-vertex pass (set 0, once)
  unsigned long long components;    // vertices that carry their own id (set 0, once)
  unsigned long long floor;         // smallest id with an out-edge (set 0, once)
};
static constexpr uint32_t CC_CW = sizeof(cc_counters) / 8;

__global__ void k_cc_init(uint32_t V, const uint32_t* __restrict__ perm, const uint32_t* __restrict__ od,
                          uint32_t* __restrict__ label, cc_counters* __restrict__ cnt) {
  uint32_t lo = 0xFFFFFFFFu;
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t id = perm ? perm[v] : (uint32_t)v;
    label[v] = id;
    if (od[v]) lo = std::min(lo, id);
  }
  for (int off = 32; off > 0; off >>= 1) lo = std::min(lo, (uint32_t)__shfl_xor((int)lo, off, 64));
  if ((threadIdx.x & 63) == 0 && lo < *(volatile unsigned long long*)&cnt->floor)
    atomicMin(&cnt->floor, (unsigned long long)lo);
}

__global__ void k_cc_zero(uint64_t* __restrict__ w, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    w[i] = 0ull;
}

__global__ void k_cc_counters(cc_counters* c) {
  c[0] = cc_counters{0, 0, 0, 0, 0, ~0ull};
  c[1] = c[2] = cc_counters{0, 0, 0, 0, 0, 0};
}

// vertices of the wave-per-vertex pass: CC_PULL_CAP < in-degree <= CC_HUB_DEG
__global__ __launch_bounds__(256) void k_cc_heavy_bits(const uint64_t* __restrict__ ptr, uint32_t V, uint64_t nwords,
                                                       uint64_t* __restrict__ bits) {
  const int lane = threadIdx.x & 63;
  for (uint64_t word = grid_wave_id(); word < nwords; word += grid_waves()) {
    const uint64_t v = word * 64 + lane;
    bool in = false;
    if (v < V) {
      const uint64_t d = ptr[v + 1] - ptr[v];
      in = d > CC_PULL_CAP && d <= CC_HUB_DEG;
    }
    const uint64_t m = __ballot(in);
    if (lane == 0) bits[word] = m;
  }
}

// one atomic per block; every thread of the block calls it
__device__ __forceinline__ void cc_add(unsigned long long act, unsigned long long* dst) {
  block_add2(act, 0, dst, dst);
}

// Push: one wave per frontier vertex u over its out-edges; a neighbour whose label is
// larger takes u's label (write_min) and becomes active.
__global__ __launch_bounds__(256) void k_cc_push(const uint32_t* __restrict__ queue, const cc_counters* cnt_in,
                                                 const uint64_t* __restrict__ ptr, const uint32_t* __restrict__ idx,
                                                 uint32_t* __restrict__ label, uint64_t* __restrict__ next_bits,
                                                 cc_counters* __restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  const uint64_t n = cnt_in->queued;
  const uint64_t wave_id = grid_wave_id(), nwaves = grid_waves();
  unsigned long long act = 0;
  for (uint64_t q = wave_id; q < n; q += nwaves) {
    const uint32_t u = queue[q];
    const uint32_t lu = label[u];  // the message's label, read when it is sent
    const uint64_t b = ptr[u], e = ptr[u + 1];
    for (uint64_t k = b + lane; k < e; k += 64) {
      const uint32_t dst = idx[k];
      if (lu < label[dst]) {
        atomicMin(&label[dst], lu);
        const uint64_t m = 1ull << (dst & 63);
        if (!(next_bits[dst >> 6] & m)) atomicOr((unsigned long long*)&next_bits[dst >> 6], (unsigned long long)m);
        ++act;
      }
    }
  }
  cc_add(act, &cnt->activated);
}

// Smallest label over the in-edges b + i0, b + i0 + step, ... below e, starting from cur, up
// to the first one at the floor.
template <bool WAVE>
__device__ __forceinline__ uint32_t cc_min(uint64_t b, uint64_t e, uint32_t i0, uint32_t step, uint32_t cur,
                                           uint32_t floor, const uint32_t* __restrict__ row_idx,
                                           const uint32_t* label) {
  for (uint64_t k0 = b; k0 < e; k0 += (uint64_t)step * CC_U) {
    uint32_t l[CC_U];
#pragma unroll
    for (int i = 0; i < CC_U; ++i) {
      const uint64_t k = k0 + (uint64_t)i * step + i0;
      l[i] = k < e ? label[row_idx[k]] : 0xFFFFFFFFu;
    }
#pragma unroll
    for (int i = 0; i < CC_U; ++i) cur = std::min(cur, l[i]);
    if (WAVE ? __ballot(cur <= floor) != 0ull : cur <= floor) break;
  }
  if (WAVE)
    for (int off = 32; off > 0; off >>= 1) cur = std::min(cur, (uint32_t)__shfl_xor((int)cur, off, 64));
  return cur;
}

// Pull for the hubs (more than CC_HUB_DEG in-edges), one chunk of in-edges per wave at
// a time: the chunk's minimum label lowers the hub's with atomicMin (several chunks of one
// hub may) and marks it.  A hub's own id is never below its label, so the chunks leave it out.
__global__ __launch_bounds__(256) void k_cc_pull_hubs(const uint64_t* __restrict__ col_ptr,
                                                      const uint32_t* __restrict__ row_idx,
                                                      const uint32_t* __restrict__ hubs,
                                                      const unsigned long long* __restrict__ nhub,
                                                      const uint64_t* __restrict__ start, uint32_t* label,
                                                      uint8_t* __restrict__ mark, const cc_counters* __restrict__ c0) {
  const int lane = threadIdx.x & 63;
  const uint64_t nwaves = grid_waves();
  const uint64_t n = *nhub;
  if (n == 0) return;
  const uint32_t floor = (uint32_t)c0->floor;
  const uint64_t total = start[n];
  for (uint64_t c = grid_wave_id(); c < total; c += nwaves) {
    uint64_t k0, k1;
    const uint32_t v = hub_chunk(col_ptr, hubs, start, n, CC_HUB_CHUNK, c, &k0, &k1);
    const uint32_t have = label[v];
    if (have <= floor) continue;
    const uint32_t cur = cc_min<true>(k0, k1, (uint32_t)lane, 64u, 0xFFFFFFFFu, floor, row_idx, label);
    if (lane == 0 && cur < have && cur < atomicMin(&label[v], cur)) mark[v] = 1;
  }
}

// Pull for the vertices of the heavy list, one wave each.
__global__ __launch_bounds__(256) void k_cc_pull_heavy(const uint64_t* __restrict__ col_ptr,
                                                       const uint32_t* __restrict__ row_idx, uint32_t* label,
                                                       const uint32_t* __restrict__ heavy, uint8_t* __restrict__ mark,
                                                       const cc_counters* __restrict__ c0) {
  const int lane = threadIdx.x & 63;
  const uint64_t n = c0->heavy, nwaves = grid_waves();
  const uint32_t floor = (uint32_t)c0->floor;
  for (uint64_t h = grid_wave_id(); h < n; h += nwaves) {
    const uint32_t v = heavy[h];
    const uint32_t have = label[v];
    if (have <= floor) continue;
    const uint32_t cur = cc_min<true>(col_ptr[v], col_ptr[v + 1], (uint32_t)lane, 64u, have, floor, row_idx, label);
    if (lane == 0 && cur < have) {
      label[v] = cur;
      mark[v] = 1;
    }
  }
}

// Pull for the others, one lane per vertex, 64 consecutive vertices per wave: the wave owns
// one word of the next bitmap, to which it adds the marks of the passes before (clearing
// them), and the epoch's counters come from these words.
// Only v's own lane, wave or chunks write label[v] in a pull epoch.
__global__ __launch_bounds__(256) void k_cc_pull(const uint64_t* __restrict__ col_ptr,
                                                 const uint32_t* __restrict__ row_idx, uint32_t V, uint64_t nwords,
                                                 const uint32_t* __restrict__ od, uint32_t* label,
                                                 uint8_t* __restrict__ mark, uint64_t* __restrict__ next_bits,
                                                 const cc_counters* __restrict__ c0, cc_counters* __restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  const uint32_t floor = (uint32_t)c0->floor;
  unsigned long long act = 0, edges = 0;
  for (uint64_t word = grid_wave_id(); word < nwords; word += grid_waves()) {
    const uint64_t v = word * 64 + lane;
    bool upd = false;
    if (v < V) {
      const uint32_t have = label[v];
      upd = mark[v] != 0;
      if (upd) mark[v] = 0;
      if (have > floor) {
        const uint64_t b = col_ptr[v], e = col_ptr[v + 1];
        if (e - b <= CC_PULL_CAP) {
          const uint32_t cur = cc_min<false>(b, e, 0u, 1u, have, floor, row_idx, label);
          if (cur < have) {
            label[v] = cur;
            upd = true;
          }
        }
      }
      if (upd) {
        act += 1;
        edges += od[v];
      }
    }
    const uint64_t m = __ballot(upd);
    if (lane == 0) next_bits[word] = m;
  }
  block_add2(act, edges, &cnt->activated, &cnt->active_edges);
}

// out-edges of the next active set (after a push), and components (label == own id: the
// smallest id that reaches a vertex is reached from no smaller one)
__global__ __launch_bounds__(256) void k_cc_active_edges(const uint64_t* __restrict__ bits, uint32_t V,
                                                         uint64_t nwords, const uint32_t* __restrict__ od,
                                                         cc_counters* __restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  unsigned long long edges = 0;
  for (uint64_t word = grid_wave_id(); word < nwords; word += grid_waves()) {
    const uint64_t w = bits[word], v = word * 64 + lane;
    if (w && v < V && ((w >> lane) & 1ull)) edges += od[v];
  }
  cc_add(edges, &cnt->active_edges);
}

__global__ __launch_bounds__(256) void k_cc_components(uint32_t V, const uint32_t* __restrict__ perm,
                                                       const uint32_t* __restrict__ label,
                                                       cc_counters* __restrict__ cnt) {
  unsigned long long n = 0;
  for (uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; v < V; v += (uint64_t)gridDim.x * blockDim.x)
    n += label[v] == (perm ? perm[v] : (uint32_t)v) ? 1u : 0u;
  cc_add(n, &cnt->components);
}

}  // namespace pe

using namespace pe;

extern "C" int pe_connected_components(pe_graph_t* g, uint32_t* labels, uint8_t* modes, uint64_t* actives,
                                       uint32_t cap, pe_cc_stats_t* stats) {
  if (!g || !labels) return PE_ERR_INVALID;
  return guarded(g->ctx, [&] {
    pe_ctx_s* ctx = g->ctx;
    hipStream_t s = ctx->stream;
    const uint32_t V = g->V;
    const uint64_t nwords = ((uint64_t)V >> 6) + 1;
    const uint32_t Vs = std::max<uint32_t>(1, V);
    dbuf<uint32_t> label(ctx, Vs), queue(ctx, Vs), heavy(ctx, std::min<uint64_t>(Vs, g->nnz / (CC_PULL_CAP + 1) + 1));
    dbuf<uint64_t> cur(ctx, nwords), nxt(ctx, nwords), marks(ctx, nwords * 8);
    dbuf<cc_counters> cnt(ctx, 3);  // set 0 holds for the whole call, the others are an epoch's
    cc_counters* c0 = cnt.p;
    const uint32_t* perm = g->relabeled ? g->perm.p : nullptr;
    const uint64_t Ep = g->directed ? g->edges : g->edges * 2;  // dualmode.hpp:261-262
    PE_HIP(hipEventRecord(ctx->t0, s));
    k_cc_counters<<<1, 1, 0, s>>>(c0);
    k_cc_init<<<grid_for(V, 256, 2048), 256, 0, s>>>(V, perm, g->od.p, label.p, c0);
    k_cc_zero<<<grid_for(nwords * 8, 256, 4096), 256, 0, s>>>(marks.p, nwords * 8);
    k_cc_heavy_bits<<<grid_for(nwords, 4, 8192), 256, 0, s>>>(g->col_ptr.p, V, nwords, cur.p);
    frontier_compact(ctx, cur.p, nwords, V, heavy.p, &c0->heavy);
    PE_HIP(hipGetLastError());
    const unsigned push_grid = persistent_grid(ctx, 1u << 20, 8);
    const unsigned pull_grid = persistent_grid(ctx, grid_for(nwords * 64, 256), 8);
    hub_table hubs;
    hub_table_build(ctx, g->col_ptr.p, V, g->nnz, CC_HUB_DEG, CC_HUB_CHUNK, hubs);
    uint64_t A = g->nnz;  // every vertex is active: the sum of all out-degrees
    uint32_t epoch = 0;
    for (uint64_t act = 1; act != 0; ++epoch) {
      const bool push = g->has_csr && ((double)A / (double)std::max<uint64_t>(Ep, 1)) < 0.05;  // dualmode.hpp:279
      cc_counters* c = c0 + 1 + (epoch & 1);
      if (push) {
        k_cc_zero<<<grid_for(nwords, 256, 4096), 256, 0, s>>>(nxt.p, nwords);
        frontier_compact(ctx, cur.p, nwords, V, queue.p, &c->queued);
        k_cc_push<<<push_grid, 256, 0, s>>>(queue.p, c, g->csr_ptr(), g->csr_idx(), label.p, nxt.p, c);
        k_cc_active_edges<<<grid_for(nwords, 4, 1024), 256, 0, s>>>(nxt.p, V, nwords, g->od.p, c);
      } else {
        uint8_t* mark = reinterpret_cast<uint8_t*>(marks.p);
        k_cc_pull_hubs<<<push_grid, 256, 0, s>>>(g->col_ptr.p, g->row_idx.p, hubs.hubs.p, hubs.count.p, hubs.start.p,
                                                 label.p, mark, c0);
        k_cc_pull_heavy<<<push_grid, 256, 0, s>>>(g->col_ptr.p, g->row_idx.p, label.p, heavy.p, mark, c0);
        k_cc_pull<<<pull_grid, 256, 0, s>>>(g->col_ptr.p, g->row_idx.p, V, nwords, g->od.p, label.p, mark, nxt.p, c0, c);
      }
      PE_HIP(hipGetLastError());
      const cc_counters* h = reinterpret_cast<const cc_counters*>(
          mail_post(ctx, reinterpret_cast<const unsigned long long*>(c), CC_CW,
                    reinterpret_cast<unsigned long long*>(c0 + 1 + ((epoch + 1) & 1)), CC_CW));
      act = h->activated;
      A = h->active_edges;
      if (epoch < cap) {
        if (modes) modes[epoch] = push ? 1 : 0;
        if (actives) actives[epoch] = act;
      }
      std::swap(cur.p, nxt.p);
      // every epoch but the last lowers a label, and labels are ids below V
      PE_REQUIRE((uint64_t)epoch <= (uint64_t)V * V + 1, PE_ERR_INTERNAL, "connected components did not terminate");
    }
    PE_HIP(hipEventRecord(ctx->t1, s));
    PE_HIP(hipEventSynchronize(ctx->t1));
    float ms = 0.f;
    PE_HIP(hipEventElapsedTime(&ms, ctx->t0, ctx->t1));
    download_external(g, label.p, labels, 4);
    if (stats) {
      stats->epochs = epoch;
      stats->seconds = ms * 1e-3;
      k_cc_components<<<grid_for(V, 256, 1024), 256, 0, s>>>(V, perm, label.p, c0);
      PE_HIP(hipGetLastError());
      stats->components = (uint32_t) reinterpret_cast<const cc_counters*>(mail_post(
          ctx, reinterpret_cast<const unsigned long long*>(c0), CC_CW, nullptr, 0))->components;
    }
  });
}
