// Triangle counting on symmetric graphs by degree orientation.
//
// The reference's TC (called at include/SSTGraph/internal/test.hpp:606)
// counts, for every stored edge (u, v) with v < u, the common neighbours of u
// and v below v (SparseMatrix.hpp:61-71 with early_end), so each triangle is
// counted once.  On a symmetric graph that count equals the number of
// triangles, which any orientation of the edges that is acyclic counts once
// as well.  This path orients each edge toward the endpoint of higher
// (degree, id) rank, so that out(u) -- the neighbours of u ranked above u --
// has at most sqrt(2m) entries, and counts |out(u) n out(v)| for every
// oriented edge u -> v: a triangle a < b < c (by rank) is found exactly once,
// at a -> b with c in both lists.
//
// The same counting kernels serve directed rows: the reference's per-edge
// count is the sum over u and v in L(u) of |L(u) n L(v)| with L(x) the ids
// of row x below x, a prefix of the sorted row, so the store itself is the
// list array there (count_list_triangles with base = off, len = lower).
//
// Layout: the oriented list of u is written at the same flat position as
// row u of the store's degree prefix (dag[prefix[u] .. + dplus[u]), sorted by
// id), so no second scan is needed.
//
// Counting stages out(u) in LDS as a hash table and streams the lists out(v),
// v in out(u), through it.  Launch tiers by |out(u)|:
//   [2, 16]    four vertices per wave
//   [17, 64], [65, 128], [129, 256], [257, 512]
//              one wave per vertex, 2 / 4 / 8 / 16 KB of table
//   > 512      one block per vertex; out(u) is hashed in tiles of 4096 ids
//              (linear probing, load <= 1/4) and every tile sees all of the
//              lists out(v).
// rMat scale 22 (134M triangles, 64M pieces of 64 ids): 7.75 ms with linear
// tables walked lane by lane, 3.37 ms now, 2.7 of it the counting, which the
// vector units' issue bounds (80% busy in the [17, 64] tier).
#include <algorithm>

#include "algo.hpp"
#include "edge_map.hpp"
#include "graph.hpp"
#include "primitives.hpp"

namespace sstg {

namespace {

constexpr uint32_t kEmpty = 0xFFFFFFFFu;  // never a vertex id (ids < n_rows)
// wave tiers: |out(u)| upper bounds (powers of two, so that the table of
// 4 * MaxOut slots holds every size table_bits() picks up to MaxOut)
constexpr uint32_t kWaveTiers = 5;
constexpr uint32_t kTierOut[kWaveTiers] = {16, 64, 128, 256, 512};
constexpr uint32_t kMidOut = kTierOut[kWaveTiers - 1];
constexpr uint32_t kBlkTile = 4096;
constexpr uint32_t kBlkTable = 4 * kBlkTile;
constexpr uint32_t kBlkChunk = 256;  // lists out(v) per block step
constexpr uint32_t kAccLanes = 64;   // spread counters, 128 B apart
constexpr uint32_t kAccStride = 16;

__device__ __forceinline__ bool ranked_above(uint32_t dv, uint32_t v,
                                             uint32_t du, uint32_t u) {
  return dv > du || (dv == du && v > u);
}

__device__ __forceinline__ uint32_t tc_hash(uint32_t x, uint32_t shift) {
  return (x * 0x9E3779B1u) >> shift;
}

// log2 of the table size for k ids: smallest power of two >= 4k, >= 64
__device__ __forceinline__ uint32_t table_bits(uint32_t k) {
  uint32_t b = 6;
  while ((1u << b) < 4 * k) b++;
  return b;
}

__device__ __forceinline__ void hash_insert(uint32_t *table, uint32_t x,
                                            uint32_t bits) {
  const uint32_t mask = (1u << bits) - 1;
  uint32_t h = tc_hash(x, 32 - bits);
  while (atomicCAS(&table[h], kEmpty, x) != kEmpty) h = (h + 1) & mask;
}

__device__ __forceinline__ uint32_t hash_has(const uint32_t *table, uint32_t x,
                                             uint32_t bits) {
  const uint32_t mask = (1u << bits) - 1;
  uint32_t h = tc_hash(x, 32 - bits);
  for (;;) {
    const uint32_t e = table[h];
    if (e == x) return 1;
    if (e == kEmpty) return 0;
    h = (h + 1) & mask;
  }
}

// Two-entry buckets: a probe is one 8-byte LDS read and two compares, with
// no loop, so a wave's 64 probes end together.  Ids beyond a bucket's two go
// to a short overflow list that every probe is compared with as well; at four
// buckets per id or more it is mostly empty (0.6 ids expected at the fullest).
// kNarrow: ids are below 2^24, so a 24-bit multiply (a quarter of the cost of
// a 32-bit one) mixes all of their bits.  The result is the bucket's byte
// offset in a table of 1 << bits buckets: drop = 29 - bits, mask = the
// offsets' bits.
template <bool kNarrow>
__device__ __forceinline__ uint32_t bucket_at(uint32_t x, uint32_t drop,
                                              uint32_t mask) {
  return ((kNarrow ? __umul24(x, 0x9E3779u) : x * 0x9E3779B1u) >> drop) & mask;
}

__device__ __forceinline__ void bucket_insert(uint2 *b, uint32_t x,
                                              uint32_t *over, uint32_t *nover) {
  if (atomicCAS(&b->x, kEmpty, x) == kEmpty) return;
  if (atomicCAS(&b->y, kEmpty, x) == kEmpty) return;
  over[atomicAdd(nover, 1u)] = x;
}

// Streams the concatenation of the lists out(v) (list j starts at dag +
// base[j], its flat range is [pre[j], pre[j+1]), pre[k] = total) through the
// hash table, P lanes striding the flat index; four loads are issued before
// their probes so that each lane keeps four gathers in flight.  A lane keeps
// its current list's end and address shift in registers and reads the LDS
// tables only when it crosses into another list.
template <uint32_t P>
__device__ __forceinline__ uint64_t probe_lists(const uint32_t *table,
                                                uint32_t bits,
                                                const uint32_t *pre,
                                                const uint64_t *base,
                                                const uint32_t *dag,
                                                uint32_t total, uint32_t me) {
  uint64_t found = 0;
  if (me >= total) return 0;
  uint32_t seg = 0, seg_start = 0, seg_end = pre[1];
  uint64_t shift = base[0];  // dag offset of flat index t: shift + t
  for (uint32_t t0 = me; t0 < total; t0 += 4 * P) {
    uint32_t w[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t t = t0 + r * P;
      w[r] = kEmpty;
      if (t < total) {
        if (seg_end <= t) {
          do {
            seg++;
            seg_start = seg_end;
            seg_end = pre[seg + 1];
          } while (seg_end <= t);
          shift = base[seg] - seg_start;  // wraps; shift + t is exact
        }
        w[r] = dag[shift + t];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (w[r] != kEmpty) found += hash_has(table, w[r], bits);
  }
  return found;
}

// Orientation, G lanes per row (rows from one degree bin).  Kept neighbours
// are written in row order by ballot rank inside the lane group.  Bound by
// the gathers of the neighbours' degrees: U of a lane's are in flight before
// the first is used (0.73 -> 0.65 ms over a rMat scale-22 graph).
template <int G, int U>
__global__ void __launch_bounds__(256)
    k_tc_orient(DevGraph g, const uint32_t *list, uint64_t count,
                const uint64_t *prefix, uint32_t *dag, uint32_t *dplus) {
  const uint64_t gid = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  const uint64_t grp = gid / G;
  const uint32_t lig = (uint32_t)(gid % G);
  if (grp >= count) return;  // whole groups leave together
  const uint32_t u = list[grp];
  const uint32_t du = g.deg[u];
  const uint32_t *row = g.pool + g.off[u];
  uint32_t *out = dag + prefix[u];
  uint32_t c = 0;
  const uint32_t lane = lane_id();
  const uint64_t gmask =
      (G == 64) ? ~0ull : (((1ull << G) - 1) << (lane & ~(uint32_t)(G - 1)));
  for (uint32_t k0 = 0; k0 < du; k0 += G * U) {
    uint32_t v[U], dv[U];
#pragma unroll
    for (int j = 0; j < U; j++) {  // past the row's end: its last entry
      const uint32_t k = k0 + j * G + lig;
      v[j] = row[k < du ? k : du - 1];
    }
#pragma unroll
    for (int j = 0; j < U; j++) dv[j] = g.deg[v[j]];
#pragma unroll
    for (int j = 0; j < U; j++) {
      const bool keep = k0 + j * G + lig < du && ranked_above(dv[j], v[j], du, u);
      if (G == 1) {
        if (keep) out[c++] = v[j];
      } else {
        const uint64_t m = __ballot(keep) & gmask;
        if (keep) out[c + mask_rank(m)] = v[j];
        c += (uint32_t)__popcll(m);
      }
    }
  }
  if (lig == 0) dplus[u] = c;
}

// NG vertices u per wave with |out(u)| <= MaxOut (NG > 1: at most 64 / NG).
// Up to 64 lists out(v) at a time are cut into pieces of 64 ids; lane t holds
// the place and length of the t-th piece, which move to scalar registers one
// piece at a time.  A piece is then one buffer load from a scalar descriptor
// whose record count ends with the list, so lanes past its end read 0 with no
// compare, address or mask of their own, and the probe is a hash, an LDS read
// and two compares: nine vector and three scalar instructions per 64 ids.
// (With a ballot, a tail mask and a length test per list, 28 scalar ones
// bounded it: 5.1 against 3.7 ms for the whole count at rMat scale 22.)  0 is no list's padding but vertex 0
// as well, so vertex 0 is kept out of the tables: rows are sorted, so it can
// only be a list's first id, and the vertices that have it look there.
template <uint32_t MaxOut, uint32_t NG, bool kNarrow>
__global__ void __launch_bounds__(64)
    k_tc_count_wave(const uint64_t *lbase, const uint32_t *lists,
                    const uint32_t *llen, const uint32_t *list,
                    uint64_t count, unsigned long long *acc) {
  static_assert((MaxOut & (MaxOut - 1)) == 0, "table size must be 2^k");
  static_assert(NG == 1 || MaxOut * NG <= 64, "a vertex's lists, one per lane");
  constexpr uint32_t L = 64 / NG;             // lanes per vertex
  constexpr uint32_t kTable = 4 * MaxOut;     // buckets per vertex
  constexpr int kPieces = 8;  // loads issued before their probes (4: 3.87 ms)
  __shared__ uint4 table4[NG * kTable / 2];
  __shared__ uint32_t over[NG][MaxOut];
  __shared__ uint32_t nover[NG];
  __shared__ uint32_t pre[64], plen[64];
  __shared__ uint64_t pbase[64];
  char *tab = reinterpret_cast<char *>(table4);
  const uint32_t lane = threadIdx.x, gi = lane / L, lig = lane % L;
  uint64_t found = 0;
  for (uint64_t i0 = (uint64_t)blockIdx.x * NG; i0 < count;
       i0 += (uint64_t)gridDim.x * NG) {  // uniform across the block
    const uint64_t i = i0 + gi;
    uint32_t d = 0;
    const uint32_t *row = lists;
    if (NG == 1 || i < count) {
      const uint32_t u = list[i];
      d = llen[u];
      row = lists + lbase[u];
    }
    // NG == 1: the table is sized to the vertex (d is uniform then)
    const uint32_t bits = NG == 1 ? table_bits(d) : __builtin_ctz(kTable);
    const uint32_t drop = 29 - bits, mask = ((1u << bits) - 1) << 3;
    const uint32_t tbase = gi * kTable * 8;
    for (uint32_t t = lane; t < (NG << bits) / 2; t += 64)
      table4[t] = make_uint4(kEmpty, kEmpty, kEmpty, kEmpty);
    if (lig == 0) nover[gi] = 0;
    __syncthreads();
    bool has0 = false;
    uint32_t hits = 0;
    for (uint32_t j0 = 0; j0 < (NG == 1 ? d : 1u); j0 += 64) {
      // this lane's list, and its id into the table
      const uint32_t j = NG == 1 ? j0 + lane : lig;
      uint32_t x = 0, len = 0;
      uint64_t base = 0;
      if (j < d) {
        x = row[j];
        len = llen[x];
        base = lbase[x];
      }
      has0 |= j == 0 && d > 0 && x == 0;
      if (NG == 1) {
        if (j0 == 0) {  // the whole table before the first probe
          has0 = __any(has0);
          for (uint32_t k = lane; k < d; k += 64) {
            const uint32_t y = k == j ? x : row[k];
            if (y)
              bucket_insert((uint2 *)(tab + bucket_at<kNarrow>(y, drop, mask)),
                            y, over[0], &nover[0]);
          }
        }
      } else {
        has0 = __shfl((int)has0, gi * L, 64);
        if (x)
          bucket_insert(
              (uint2 *)(tab + tbase + bucket_at<kNarrow>(x, drop, mask)), x,
              over[gi], &nover[gi]);
      }
      if (has0 && len && lists[base] == 0) hits++;
      const uint32_t mine = (len + 63) / 64;
      const uint32_t incl = wave_inclusive_sum(mine);
      const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
      pre[lane] = incl - mine;
      plen[lane] = len;
      pbase[lane] = base;
      __syncthreads();
      uint32_t any_over = 0;
#pragma unroll
      for (uint32_t k = 0; k < NG; k++) any_over |= nover[k];
      any_over = __builtin_amdgcn_readfirstlane(any_over);
      for (uint32_t t0 = 0; t0 < total; t0 += 64) {
        // the lane's piece: the last list that starts at or before it
        const uint32_t t = t0 + lane;
        uint32_t s = 0;
#pragma unroll
        for (uint32_t step = 32; step > 0; step >>= 1)
          if (pre[s + step] <= t) s += step;
        const uint32_t off = (t - pre[s]) * 64;
        const uint64_t place = t < total ? (uint64_t)(lists + pbase[s] + off) : 0;
        const uint32_t bytes = t < total ? (plen[s] - off) * 4 : 0;
        const uint32_t here = total - t0 < 64 ? total - t0 : 64;
        for (uint32_t p = 0; p < here; p += kPieces) {
          uint32_t w[kPieces], grp[kPieces];
#pragma unroll
          for (int k = 0; k < kPieces; k++) {  // pieces past the last are empty
            const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)place, p + k);
            const uint32_t hi =
                __builtin_amdgcn_readlane((uint32_t)(place >> 32), p + k);
            const uint32_t nb = __builtin_amdgcn_readlane(bytes, p + k);
            if (NG > 1) grp[k] = __builtin_amdgcn_readlane(s / L, p + k);
            w[k] = __builtin_amdgcn_raw_buffer_load_b32(
                __builtin_amdgcn_make_buffer_rsrc(
                    (void *)(((uint64_t)hi << 32) | lo), 0, (int)nb, 0x00020000),
                (int)(lane * 4), 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);  // every load before any wait
          uint2 e[kPieces];
#pragma unroll
          for (int k = 0; k < kPieces; k++) {
            uint32_t at = bucket_at<kNarrow>(w[k], drop, mask);
            if (NG > 1) at |= grp[k] * (kTable * 8);
            e[k] = *(const uint2 *)(tab + at);
          }
#pragma unroll
          for (int k = 0; k < kPieces; k++)
            hits += (uint32_t)(e[k].x == w[k]) | (uint32_t)(e[k].y == w[k]);
          if (any_over)
#pragma unroll
            for (int k = 0; k < kPieces; k++) {
              const uint32_t g = NG > 1 ? grp[k] : 0;
              for (uint32_t o = 0; o < nover[g]; o++)
                hits += over[g][o] == w[k] ? 1u : 0u;
            }
        }
      }
      __syncthreads();  // pre, plen and pbase are rewritten
    }
    found += hits;
    __syncthreads();  // the tables are reused by the next vertices
  }
  found = wave_sum(found);
  if (lane == 0 && found)
    atomicAdd(&acc[(blockIdx.x % kAccLanes) * kAccStride],
              (unsigned long long)found);
}

// One block of 256 per vertex u with |out(u)| > kMidOut: out(u) is hashed in
// tiles of kBlkTile ids; for each tile every list out(v), v in out(u), is
// streamed through it in steps of kBlkChunk lists.
__global__ void __launch_bounds__(256)
    k_tc_count_block(const uint64_t *lbase, const uint32_t *lists,
                     const uint32_t *llen, const uint32_t *list,
                     uint64_t count, unsigned long long *acc) {
  __shared__ uint32_t table[kBlkTable];
  __shared__ uint32_t pre[kBlkChunk + 1];
  __shared__ uint64_t base[kBlkChunk];
  const uint32_t tid = threadIdx.x;
  uint64_t found = 0;
  for (uint64_t i = blockIdx.x; i < count; i += gridDim.x) {
    const uint32_t u = list[i];
    const uint32_t d = llen[u];
    const uint32_t *row = lists + lbase[u];
    for (uint32_t t0 = 0; t0 < d; t0 += kBlkTile) {
      const uint32_t tn = (d - t0) < kBlkTile ? (d - t0) : kBlkTile;
      const uint32_t bits = table_bits(tn);
      for (uint32_t t = tid; t < (1u << bits); t += 256) table[t] = kEmpty;
      __syncthreads();
      for (uint32_t j = tid; j < tn; j += 256) hash_insert(table, row[t0 + j], bits);
      __syncthreads();
      for (uint32_t c0 = 0; c0 < d; c0 += kBlkChunk) {
        const uint32_t cn = (d - c0) < kBlkChunk ? (d - c0) : kBlkChunk;
        uint32_t len = 0;
        if (tid < cn) {
          const uint32_t x = row[c0 + tid];
          len = llen[x];
          base[tid] = lbase[x];
        }
        uint32_t total = 0;
        const uint32_t off = em::block_scan_u32(len, &total);
        if (tid < cn) pre[tid] = off;
        if (tid == 0) pre[cn] = total;
        __syncthreads();
        found += probe_lists<256>(table, bits, pre, base, lists, total, tid);
        __syncthreads();  // pre and base are rewritten by the next step
      }
    }
  }
  found = wave_sum(found);
  if ((tid & 63) == 0 && found)
    atomicAdd(&acc[(blockIdx.x % kAccLanes) * kAccStride],
              (unsigned long long)found);
}

// acc[i * kAccStride] for i < kAccLanes are the spread counters
__global__ void k_tc_acc_clear(unsigned long long *acc) {
  acc[threadIdx.x * kAccStride] = 0;
}

__global__ void k_tc_acc_sum(unsigned long long *acc) {
  uint64_t v = acc[threadIdx.x * kAccStride];
  v = wave_sum(v);
  if (threadIdx.x == 0) acc[0] = v;
}

// Triangles of a graph whose every edge has its reverse that contain at
// least one changed undirected edge, each counted once, by its smallest
// changed edge in (min << 32 | max) order.  keys: the changed pairs, sorted,
// with both directions of every edge.  One wave per changed edge {u, v},
// u < v: lanes take the ids of the shorter row and look each up in the
// longer one; a common neighbour w counts unless {u, w} or {v, w} is also
// changed with a smaller key.  Per-block partial sums, no atomics.
__device__ __forceinline__ bool sorted_has(const uint64_t *a, uint64_t n,
                                           uint64_t x) {
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (a[mid] < x)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo < n && a[lo] == x;
}

__global__ void __launch_bounds__(256)
    k_tc_delta(DevGraph g, const uint64_t *keys, uint64_t count,
               unsigned long long *part) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t waves = (uint64_t)gridDim.x * 4;
  uint64_t found = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * 4 + threadIdx.x / 64; i < count;
       i += waves) {
    const uint64_t kuv = keys[i];
    const uint32_t u = (uint32_t)(kuv >> 32), v = (uint32_t)kuv;
    if (u >= v) continue;  // the wave's edge: each undirected edge once
    const uint32_t du = g.deg[u], dv = g.deg[v];
    const uint32_t a = du <= dv ? u : v, b = du <= dv ? v : u;
    const uint32_t da = du <= dv ? du : dv, db = du <= dv ? dv : du;
    const uint32_t *ra = g.pool + g.off[a], *rb = g.pool + g.off[b];
    for (uint32_t j = lane; j < da; j += 64) {
      const uint32_t w = ra[j];
      if (w == u || w == v) continue;
      if (!row_has(rb, db, w)) continue;
      const uint64_t kuw = u < w ? ((uint64_t)u << 32) | w
                                 : ((uint64_t)w << 32) | u;
      const uint64_t kvw = v < w ? ((uint64_t)v << 32) | w
                                 : ((uint64_t)w << 32) | v;
      if (kuw < kuv && sorted_has(keys, count, kuw)) continue;
      if (kvw < kuv && sorted_has(keys, count, kvw)) continue;
      found++;
    }
  }
  __shared__ unsigned long long wsum[4];
  found = wave_sum(found);
  if (lane == 0) wsum[threadIdx.x / 64] = found;
  __syncthreads();
  if (threadIdx.x == 0)
    part[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

__global__ void __launch_bounds__(256)
    k_tc_delta_sum(const unsigned long long *part, uint32_t nb,
                   unsigned long long *out) {
  unsigned long long t = 0;
  for (uint32_t i = threadIdx.x; i < nb; i += 256) t += part[i];
  __shared__ unsigned long long wsum[4];
  t = wave_sum(t);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x / 64] = t;
  __syncthreads();
  if (threadIdx.x == 0) *out = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

uint32_t grid_for(uint64_t count) {
  return (uint32_t)(count < (1u << 24) ? count : (1u << 24));
}

// The counting kernel of tier c over the cnt vertices of l.
template <bool kNarrow>
void launch_tier(uint32_t c, uint64_t cnt, hipStream_t s, const uint64_t *lbase,
                 const uint32_t *lists, const uint32_t *llen, const uint32_t *l,
                 unsigned long long *acc) {
  const uint32_t grid = grid_for(cnt);
  switch (c) {
    case 0:
      SSTG_LAUNCH((k_tc_count_wave<kTierOut[0], 4, kNarrow>),
                  grid_for(ceil_div(cnt, 4)), 64, 0, s, lbase, lists, llen, l,
                  cnt, acc);
      break;
    case 1:
      SSTG_LAUNCH((k_tc_count_wave<kTierOut[1], 1, kNarrow>), grid, 64, 0, s,
                  lbase, lists, llen, l, cnt, acc);
      break;
    case 2:
      SSTG_LAUNCH((k_tc_count_wave<kTierOut[2], 1, kNarrow>), grid, 64, 0, s,
                  lbase, lists, llen, l, cnt, acc);
      break;
    case 3:
      SSTG_LAUNCH((k_tc_count_wave<kTierOut[3], 1, kNarrow>), grid, 64, 0, s,
                  lbase, lists, llen, l, cnt, acc);
      break;
    case 4:
      SSTG_LAUNCH((k_tc_count_wave<kTierOut[4], 1, kNarrow>), grid, 64, 0, s,
                  lbase, lists, llen, l, cnt, acc);
      break;
    default:
      SSTG_LAUNCH(k_tc_count_block, grid, 256, 0, s, lbase, lists, llen, l, cnt,
                  acc);
  }
}

}  // namespace

int count_list_triangles(sstg_graph *g, const uint64_t *lbase,
                         const uint32_t *lists, const uint32_t *llen,
                         uint64_t *out) {
  hipStream_t s = g->stream;
  const uint32_t n = g->n_rows;
  uint32_t *list = nullptr;
  unsigned long long *acc = nullptr;
  SSTG_TRY(g->ws.get(kWsTcList, n, &list));
  SSTG_TRY(g->ws.get(kWsTcAcc, kAccLanes * kAccStride, &acc));
  SSTG_LAUNCH(k_tc_acc_clear, 1, kAccLanes, 0, s, acc);
  uint32_t hi[kWaveTiers + 1];
  for (uint32_t c = 0; c < kWaveTiers; c++) hi[c] = kTierOut[c];
  hi[kWaveTiers] = 0xFFFFFFFFu;
  uint64_t cnts[kWaveTiers + 1], longest = 0;
  SSTG_TRY(graph_bins(g, llen, 2, hi, kWaveTiers + 1, list, cnts, &longest));
  // the flat probe index of one vertex (up to 512 lists, or 256 per block
  // step) is 32-bit: lists of 2^23 ids or more go to the caller's fallback
  if (longest >= (1u << 23)) return SSTG_E_UNSUPPORTED;
  const uint32_t *l = list;
  for (uint32_t c = 0; c <= kWaveTiers; l += cnts[c], c++) {
    const uint64_t cnt = cnts[c];
    if (!cnt) continue;
    if (n <= (1u << 24))
      launch_tier<true>(c, cnt, s, lbase, lists, llen, l, acc);
    else
      launch_tier<false>(c, cnt, s, lbase, lists, llen, l, acc);
  }
  SSTG_LAUNCH(k_tc_acc_sum, 1, kAccLanes, 0, s, acc);
  SSTG_HIP(hipMemcpyAsync(g->host_rb, acc, sizeof(uint64_t),
                          hipMemcpyDeviceToHost, s));
  SSTG_HIP(hipStreamSynchronize(s));
  *out = g->host_rb[0];
  return SSTG_OK;
}

int tc_oriented(sstg_graph *g, uint64_t *out) {
  hipStream_t s = g->stream;
  const uint32_t n = g->n_rows;
  DegreeBins bins;
  SSTG_TRY(degree_bins(g, &bins));
  const uint64_t *prefix = nullptr;
  SSTG_TRY(graph_degree_prefix(g, &prefix));
  uint32_t *dag = nullptr, *dplus = nullptr;
  SSTG_TRY(g->ws.get(kWsTcDag, g->m, &dag));
  SSTG_TRY(g->ws.get(kWsTcDplus, n, &dplus));
  const DevGraph v = g->view();
  if (bins.count[0])
    SSTG_LAUNCH((k_tc_orient<1, 4>), ceil_div(bins.count[0], 256), 256, 0, s, v,
                (const uint32_t *)bins.list[0], bins.count[0], prefix, dag,
                dplus);
  if (bins.count[1])
    SSTG_LAUNCH((k_tc_orient<8, 4>), ceil_div(bins.count[1] * 8, 256), 256, 0, s, v,
                (const uint32_t *)bins.list[1], bins.count[1], prefix, dag,
                dplus);
  for (int b = 2; b < 4; b++)
    if (bins.count[b])
      SSTG_LAUNCH((k_tc_orient<64, 4>), ceil_div(bins.count[b] * 64, 256), 256, 0,
                  s, v, (const uint32_t *)bins.list[b], bins.count[b], prefix,
                  dag, dplus);
  return count_list_triangles(g, prefix, dag, dplus, out);
}

int tc_delta(sstg_graph *g, const uint64_t *keys, uint64_t count,
             uint64_t *out) {
  *out = 0;
  if (count == 0) return SSTG_OK;
  hipStream_t s = g->stream;
  const uint32_t nb = (uint32_t)std::min<uint64_t>(4096, (count + 7) / 8);
  unsigned long long *part = nullptr;
  SSTG_TRY(g->ws.get(kWsTcDelta, nb + 1, &part));
  SSTG_LAUNCH(k_tc_delta, nb, 256, 0, s, g->view(), keys, count, part);
  SSTG_LAUNCH(k_tc_delta_sum, 1, 256, 0, s, (const unsigned long long *)part,
              nb, part + nb);
  SSTG_HIP(hipMemcpyAsync(g->host_rb + 40, part + nb, sizeof(uint64_t),
                          hipMemcpyDeviceToHost, s));
  SSTG_HIP(hipStreamSynchronize(s));
  *out = g->host_rb[40];
  return SSTG_OK;
}

}  // namespace sstg
