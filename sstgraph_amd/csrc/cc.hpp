// Connected components by union-find on the device store, shared by the
// single-graph CC (algo.hip) and the many-graph pass (multi.hip).
//
// The reference's harness only uses the partition CC returns
// (internal/test.hpp:571-601); labels here are the smallest vertex id of each
// component.  The forest always hooks the larger slot under the smaller
// (p[x] <= x throughout, so every root is its tree's smallest slot).
//
// Symmetric graphs first merge most vertices into one component without a
// compare-and-swap: every vertex hooks to the neighbour at one end of its row
// (a plain store into its own slot), and then in each sampling round every
// tree's root takes the smallest root met through its members' sampled
// neighbours (an atomic minimum that nothing waits for or retries).  A
// minimum that replaces another candidate drops that link, which costs
// nothing but a later merge: the rounds are only a head start.  The most
// common root among 64 samples per graph is then taken as that graph's large
// component, and the vertices outside it link all of their edges with
// compare-and-swap.  A skipped edge (v, w) with v inside the large component
// is linked from w's side, because w's row holds v; if w is inside too, the
// edge joins nothing new.  Rows without their reverses link every stored
// edge.
//
// What bounds it is one cache line per row (the first hook), then gathers of
// p, one line each, for the vertices not yet in the large tree, and above all
// same-address atomics on the roots that many vertices want to lower.  Hence:
//   - The first hook takes the end of the row where the hubs are: each vertex
//     without a neighbour beyond it on that side leaves a tree, and those are
//     few where the ids on that side have many neighbours.  So slots run
//     against the ids in a graph whose upper ids hold most edges (see Slots),
//     and such a graph's labels take one more pass.  At rMat scale 24 (hubs
//     at the top) hooking to the first neighbour leaves 1.06 ms of rounds and
//     linking, to the last 0.39 ms plus 0.09 ms for the labels.
//   - A round, and the linking, run a sixteenth of the vertices in a launch
//     of their own: the rest then read roots that are already low and stay
//     silent (Erdos-Renyi, 262K vertices of degree 16: 340 -> 105 us).
// CC at rMat scale 24: 2.0-2.4 ms when every vertex linked two neighbours
// with compare-and-swap, 1.05 ms now, of which the first hook (every row's
// line, 1.6 GB at 4.7 TB/s) is 0.34 ms.
#pragma once

#include "graph.hpp"

namespace sstg {
namespace cc {
namespace {  // internal linkage: included by several files

constexpr int kT = 256;
// two: a third costs 0.1 ms at rMat scale 24 and saves 0.24 ms only on sparse
// even graphs (4M Erdos-Renyi vertices of degree 12)
constexpr uint32_t kHookRounds = 2;
constexpr uint32_t kInfRoot = 0xFFFFFFFFu;  // no vertex: ids are below n

__device__ __forceinline__ uint32_t find(uint32_t *p, uint32_t x) {
  uint32_t y = p[x];
  while (y != x) {
    uint32_t z = p[y];
    if (z != y) p[x] = z;  // path halving; only ever lowers p[x]
    x = y;
    y = z;
  }
  return x;
}

// union of the sets of u and w: the larger root is hooked under the smaller
__device__ __forceinline__ void link(uint32_t *p, uint32_t u, uint32_t w) {
  uint32_t ru = find(p, u), rw = find(p, w);
  while (ru != rw) {
    const uint32_t hi = ru > rw ? ru : rw, lo = ru > rw ? rw : ru;
    const uint32_t old = atomicCAS(&p[hi], hi, lo);
    if (old == hi) break;
    ru = find(p, old);
    rw = find(p, lo);
  }
}

__device__ __forceinline__ uint32_t sample_hash(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

// The forest's numbering of a graph's vertices: its ids, or against them
// (lo + hi - 1 - v over the graph's range [lo, hi)) where the upper half of
// the ids holds more than 5/8 of the edges, as in the reference's rMat, whose
// hubs have mostly 1 bits.  A graph with its edges spread evenly keeps its
// ids: it gains nothing from a second pass over the labels.
struct Slots {
  const uint64_t *prefix;  // degree prefix
  const uint32_t *vbase, *graph_of;  // null: one graph of n vertices
  uint32_t n;
  __device__ __forceinline__ bool against(uint32_t v, uint32_t *ends) const {
    uint32_t lo = 0, hi = n;
    if (graph_of) {
      const uint32_t gi = graph_of[v];
      lo = vbase[gi];
      hi = vbase[gi + 1];
    }
    const uint64_t a = prefix[lo], m = prefix[lo + (hi - lo) / 2],
                   b = prefix[hi];
    *ends = lo + hi - 1u;  // ids are below 2^32 - 1; the sum may wrap
    return 8 * (b - m) > 5 * (b - a);
  }
};

// p[v] = min(v, first neighbour): rows are sorted, so this is a link
// without atomics (the start of the every-edge schedule)
__global__ void k_init(DevGraph g, uint32_t *p) {
  const uint64_t v = (uint64_t)blockIdx.x * kT + threadIdx.x;
  if (v >= g.n) return;
  uint32_t m = (uint32_t)v;
  if (g.deg[v]) {
    const uint32_t first = g.pool[g.off[v]];
    if (first < m) m = first;
  }
  p[v] = m;
}

// Each slot hooks to its vertex's neighbour of the smallest slot (the row's
// first or last), and the neighbours' slots at kHookRounds hashed row
// positions go to samples[r * n + slot] (the slot itself where the row is
// empty): they mostly share that cache line, so the sampling rounds read no
// row again.
//
// Hooks inside a block are followed to their end in LDS, by doubling: where
// ids run along the edges (paths, ladders, narrow grids) these hooks chain
// whole components, and walking the chains was 1 us per 20 vertices.  CC of a
// path of 4M vertices 4.9 -> 0.21 ms, of 20,000 0.95 -> 0.06, of a 4096 x 4096
// grid 1.19 -> 0.52; rMat scale 24 stays at 0.97, most of its hooks leaving
// the block.  Windows of 1024 to 4096 in the compression as well: no gain.
__global__ void __launch_bounds__(kT)
    k_hook_ends(DevGraph g, Slots sl, uint32_t *p, uint32_t *samples) {
  __shared__ uint32_t up[kT];
  const uint64_t v0 = (uint64_t)blockIdx.x * kT, v = v0 + threadIdx.x;
  const bool in = v < g.n;
  uint32_t ends = 0, to = (uint32_t)v;  // the vertex hooked to
  bool against = false;
  if (in) {
    against = sl.against((uint32_t)v, &ends);
    const uint32_t x = against ? ends - (uint32_t)v : (uint32_t)v;
    uint32_t s[kHookRounds];
#pragma unroll
    for (uint32_t r = 0; r < kHookRounds; r++) s[r] = x;
    const uint32_t d = g.deg[v];
    if (d) {
      const uint32_t *row = g.pool + g.off[v];
      const uint32_t e = row[against ? d - 1 : 0];
      const uint32_t h = sample_hash((uint32_t)v);
#pragma unroll
      for (uint32_t r = 0; r < kHookRounds; r++) {
        const uint32_t w = row[(h + r) % d];
        s[r] = against ? ends - w : w;
      }
      to = against ? max(to, e) : min(to, e);
    }
#pragma unroll
    for (uint32_t r = 0; r < kHookRounds; r++)
      samples[r * (uint64_t)g.n + x] = s[r];
  }
  up[threadIdx.x] = to;
  __syncthreads();
  for (;;) {  // uniform
    const uint64_t l = to - v0;  // wraps below the block
    const uint32_t next = l < kT ? up[l] : to;
    if (!__syncthreads_or(next != to)) break;
    up[threadIdx.x] = to = next;
    __syncthreads();
  }
  if (in) p[against ? ends - (uint32_t)v : (uint32_t)v] = against ? ends - to : to;
}

// One sampling round: the larger of the roots of v and its sampled neighbour
// takes the smaller if that is below its parent (so p[x] <= x holds and no
// cycle forms whatever the order).  With giant given the forest is compressed
// and members of their graph's largest tree so far leave at once: an edge out
// of it is also its other end's, and the gather of p[w] is what the round
// costs.
__global__ void k_hook(uint32_t v0, uint32_t n, uint32_t *p,
                       const uint32_t *sample, const uint32_t *giant,
                       const uint32_t *graph_of) {
  const uint64_t v = v0 + (uint64_t)blockIdx.x * kT + threadIdx.x;
  if (v >= n) return;
  uint32_t a = p[v];
  if (giant && a == giant[graph_of ? graph_of[v] : 0u]) return;
  const uint32_t w = sample[v];
  if (w == (uint32_t)v) return;
  uint32_t b = p[w];
  if (!giant) {
    a = find(p, a);
    b = find(p, b);
  }
  const uint32_t hi = a > b ? a : b, lo = a > b ? b : a;
  if (hi != lo && p[hi] > lo) atomicMin(&p[hi], lo);
}

__global__ void k_compress(uint32_t n, uint32_t *p) {
  const uint64_t v = (uint64_t)blockIdx.x * kT + threadIdx.x;
  if (v >= n) return;
  p[v] = find(p, (uint32_t)v);
}

// giant[i] = the most common root among 64 sampled vertices of graph i
// (vertices [vbase[i], vbase[i+1]), or [0, n) when vbase is null); one wave
// per graph, ties to the lowest sampled lane.  Positions are hashed: evenly
// spaced ids share their low bits, and in rMat graphs ids with many zero bits
// are mostly isolated.
__global__ void k_mode(const uint32_t *vbase, uint32_t graphs, uint32_t n,
                       uint32_t *p, uint32_t *giant) {
  const uint64_t gi = ((uint64_t)blockIdx.x * kT + threadIdx.x) / kWave;
  const uint32_t lane = lane_id();
  if (gi >= graphs) return;  // whole waves leave together
  const uint32_t b = vbase ? vbase[gi] : 0u;
  const uint32_t e = vbase ? vbase[gi + 1] : n;
  const uint32_t len = e - b;
  uint32_t r = kInfRoot;
  if (len)
    r = find(p, b + sample_hash((uint32_t)gi * kWave + lane + 1u) % len);
  uint32_t best = 0, best_r = kInfRoot;
  for (int l = 0; l < kWave; l++) {
    const uint32_t x = __shfl(r, l, kWave);
    uint32_t c = (uint32_t)__popcll(__ballot(x != kInfRoot && r == x));
    if (c > best) {
      best = c;
      best_r = x;
    }
  }
  if (lane == 0) giant[gi] = best_r;
}

// Every edge of the vertices outside their graph's large component.  Where
// slots run against the ids, low is reset for k_low: an isolated vertex is
// its own label.
__global__ void k_link_rest(DevGraph g, Slots sl, uint32_t v0, uint32_t v1,
                            uint32_t *p, const uint32_t *giant, uint32_t *low) {
  const uint64_t v = v0 + (uint64_t)blockIdx.x * kT + threadIdx.x;
  if (v >= v1) return;
  uint32_t ends;
  const bool against = sl.against((uint32_t)v, &ends);
  const uint32_t x = against ? ends - (uint32_t)v : (uint32_t)v;
  const uint32_t d = g.deg[v];
  if (against) low[x] = d ? kInfRoot : (uint32_t)v;
  if (d == 0) return;
  // inside the large component now: its edges are linked from the other
  // side or join nothing new (compression races can leave p[x] one hop
  // short of the root, so roots are compared, not p[x])
  const uint32_t c = giant[sl.graph_of ? sl.graph_of[v] : 0u];
  if (find(p, x) == find(p, c)) return;
  const uint32_t *row = g.pool + g.off[v];
  for (uint32_t k = 0; k < d; k++)
    link(p, x, against ? ends - row[k] : row[k]);
}

// low[root] = the smallest id of each component of the vertices [v0, v1)
// where slots run against the ids.  A wave's ids ascend, so the first lane of
// each root speaks for the others, and it stays silent once a smaller id is
// there.  (Same-address atomics queue: the caller runs the first ids in a
// launch of their own, after which a large component's waves find theirs.)
__global__ void __launch_bounds__(kT)
    k_low(Slots sl, uint32_t v0, uint32_t v1, uint32_t *p, uint32_t *low) {
  const uint64_t v = v0 + (uint64_t)blockIdx.x * kT + threadIdx.x;
  uint32_t ends, root = kInfRoot;
  if (v < v1 && sl.against((uint32_t)v, &ends))
    root = find(p, ends - (uint32_t)v);
  uint64_t todo =
      __ballot(root != kInfRoot && low[root != kInfRoot ? root : 0u] > (uint32_t)v);
  while (todo) {  // uniform across the wave
    const uint32_t first = (uint32_t)__ffsll((unsigned long long)todo) - 1;
    const uint32_t r = __shfl(root, first, kWave);
    if (lane_id() == first) atomicMin(&low[r], (uint32_t)v);
    todo &= ~__ballot(root == r);
  }
}

// The label of vertex v: the smallest id of its component.
__device__ __forceinline__ uint32_t label_of(const Slots &sl, uint32_t v,
                                             uint32_t *p, const uint32_t *low) {
  uint32_t ends;
  return sl.against(v, &ends) ? low[find(p, ends - v)] : find(p, v);
}

// every stored edge, flat over edges (8 per thread)
__global__ void k_hook_all(DevGraph g, const uint64_t *prefix, uint64_t m,
                           uint32_t *p) {
  uint64_t e = ((uint64_t)blockIdx.x * kT + threadIdx.x) * 8;
  if (e >= m) return;
  const uint64_t end = e + 8 < m ? e + 8 : m;
  uint64_t v = find_segment(prefix, g.n, e);
  for (; e < end; e++) {
    while (e >= prefix[v + 1]) v++;
    link(p, (uint32_t)v, g.pool[g.off[v] + (e - prefix[v])]);
  }
}

// Vertices below which the first launch of k_low covers all.
constexpr uint32_t kLowFirst = 1u << 16;
// Below kCompressMin vertices p fits an L2 several times over and a launch
// costs more than the hops it saves, so the rounds find their roots
// themselves (rMat scale 16: 83 -> 72 us; scale 18: 93 -> 95 us).
constexpr uint32_t kCompressMin = 1u << 17;
// The first launch of a round takes 1 / kHookFirst of the vertices (1 / 64:
// 251 against 193 us at 1M Erdos-Renyi vertices of degree 16), from kSplitMin
// vertices on (65K such vertices: 182 -> 78 us, 4K: 41 -> 58 us).
constexpr uint32_t kHookFirst = 16;
constexpr uint32_t kSplitMin = 1u << 14;

// The forest of symmetric graphs into p, the large component of each of
// `graphs` graphs into giant; afterwards label_of gives the labels, with
// samples (kHookRounds * n entries) as its `low`.  Launches only, so a caller
// may be recording the stream.
inline int forest_symmetric(const DevGraph &g, const Slots &sl, uint32_t *p,
                            uint32_t *samples, uint32_t graphs,
                            uint32_t *giant, hipStream_t s) {
  if (g.n == 0) return SSTG_OK;
  const uint64_t nb = ceil_div(g.n, kT);
  SSTG_LAUNCH(k_hook_ends, nb, kT, 0, s, g, sl, p, samples);
  const bool small = g.n < kCompressMin;
  const uint32_t cut[3] = {0, g.n < kSplitMin ? g.n : g.n / kHookFirst, g.n};
  const uint64_t mode_blocks = ceil_div((uint64_t)graphs * kWave, kT);
  for (uint32_t r = 0; r < kHookRounds; r++) {
    if (!small) {
      SSTG_LAUNCH(k_compress, nb, kT, 0, s, g.n, p);
      SSTG_LAUNCH(k_mode, mode_blocks, kT, 0, s, sl.vbase, graphs, g.n, p,
                  giant);
    }
    // slots and ids of a graph fill the same range, so graph_of serves both
    for (int h = 0; h < 2 && cut[h] < g.n; h++)
      SSTG_LAUNCH(k_hook, ceil_div(cut[h + 1] - cut[h], kT), kT, 0, s, cut[h],
                  cut[h + 1], p,
                  (const uint32_t *)(samples + r * (uint64_t)g.n),
                  small ? (const uint32_t *)nullptr : (const uint32_t *)giant,
                  sl.graph_of);
  }
  if (!small) SSTG_LAUNCH(k_compress, nb, kT, 0, s, g.n, p);
  SSTG_LAUNCH(k_mode, mode_blocks, kT, 0, s, sl.vbase, graphs, g.n, p, giant);
  for (int h = 0; h < 2 && cut[h] < g.n; h++)
    SSTG_LAUNCH(k_link_rest, ceil_div(cut[h + 1] - cut[h], kT), kT, 0, s, g,
                sl, cut[h], cut[h + 1], p, (const uint32_t *)giant, samples);
  const uint32_t first = g.n < kLowFirst ? g.n : kLowFirst;
  SSTG_LAUNCH(k_low, ceil_div(first, kT), kT, 0, s, sl, 0u, first, p, samples);
  if (g.n > first)
    SSTG_LAUNCH(k_low, ceil_div(g.n - first, kT), kT, 0, s, sl, first, g.n, p,
                samples);
  return SSTG_OK;
}

}  // namespace
}  // namespace cc
}  // namespace sstg
