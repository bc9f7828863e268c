// ct_gather.hip -- box and segment queries, one wavefront for a few queries (ct_gather.h has the walk).
//
// What bounds it: the latency of a step's loads (a node record, a cell box, a clip's vertices), hidden by
// the 16 to 20 wavefronts a CU holds (LDS, registers); the FP64 arithmetic of the segment tests is
// about half of the segments' time.  1e6 queries on a million-cell mesh, before (subqueries, one lane
// each, and their replay and sort kernels) and now, whole calls: boxes (31.6e6 rows) 1.94 and 1.20 ms,
// segments (13.6e6 rows) 3.50 and 2.40 ms; 2e3 segments 560 and 100 us.
//
// Rows go to a pool (each wavefront allocates from one of several counters); an exclusive scan of
// the counts gives the output offsets, and the copy kernels write whole output lines in query order.
// A query with more hits than the LDS lists hold, or that the pool has no room for, is left to the
// caller (starts[q] = -1): few go to ct_long.hip, a wavefront each, many to the subqueries (ct_split.hip).
#include <algorithm>
#include <cmath>

#include "ct_gather.h"

namespace ct {
namespace {

// Workgroups go round-robin over the 8 XCDs (workgroup b runs on XCD b % 8).  Workgroup b takes block
// block_of(b): every XCD sweeps whole chunks of kXcdChunk consecutive blocks, chunk c on XCD c % 8, so
// that its L2 holds the part of the tree its queries (in Morton order) share, while all XCDs
// stay within the same stretch of the order.  Measured against the plain order with the heaviest
// queries first, 1e6 queries: boxes 1.31 and 1.22 ms, segments 2.80 and 2.67; chunks of 32 blocks:
// 1.24 and 2.71; of 512: 1.23 and 2.68.
constexpr int kXcds = 8, kXcdChunk = 128;

__device__ __forceinline__ int64_t block_of(unsigned b) {
  const unsigned x = b % kXcds, j = b / kXcds;
  return ((int64_t)(j / kXcdChunk) * kXcds + x) * kXcdChunk + j % kXcdChunk;
}

inline unsigned gather_grid(int64_t blocks) {
  const int64_t round = kXcds * kXcdChunk;
  return (unsigned)((blocks + round - 1) / round * round);
}

// One block of queries per workgroup, one wavefront each: the hardware's scheduler balances them.  Faces of
// more than 8 vertices: two wavefronts a SIMD, with spills (1e5 segments on 12-gons 1008 us with one and
// none, 660 with two; on 24-gons 1461 and 1041).
template <int KIND, int MAXV>
__global__ void __launch_bounds__(64, MAXV <= 8 ? 4 : 2)
k_gather(TreeView t, const double* __restrict__ qs, const int32_t* __restrict__ order, int64_t n, GatherParams p,
         Pool pool, int64_t* __restrict__ counts, int64_t* __restrict__ starts, int64_t* tail) {
  const int64_t i0 = block_of(blockIdx.x) * p.per_wave;
  if (i0 >= n) return;
  PoolRows rows;
  rows.sub = (int)(blockIdx.x % (unsigned)pool.counters);
  gather_block<KIND, MAXV>(t, qs, order, i0, (int)min((int64_t)p.per_wave, n - i0), p, pool, rows, counts, starts, tail);
}

// The queries left to the caller (starts < 0), one list entry each; the lanes of a wavefront in order.
__global__ void __launch_bounds__(kBlock) k_left(int64_t n, const int64_t* __restrict__ starts, int32_t* __restrict__ left,
                                                 int64_t room, unsigned long long* __restrict__ found) {
  const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool is = q < n && starts[q] < 0;
  const uint64_t mask = __ballot(is);
  if (!mask) return;
  const int lead = __ffsll((unsigned long long)mask) - 1;
  unsigned long long at = 0;
  if (lane_id() == lead) at = atomicAdd(found, (unsigned long long)__popcll(mask));
  at = __shfl(at, lead) + below(mask);
  if (is && (int64_t)at < room) left[at] = (int32_t)q;
}

// Output rows from the pool, `per_wave` queries per wavefront (a power of two, at most 64; fewer when
// there are few: 2e3 segments in 32 wavefronts took 18 us, a query each 5) in query order: their rows are one run of
// the output, written 64 rows per step (row g's owner by a binary search over the wavefront's
// prefix), so every output line is written whole.  kAhead steps run together: a row is a chain of two
// or three loads.  Queries whose rows end past `capacity` are left out.
constexpr int kAhead = 4;
constexpr int64_t kRowWaves = 4096;

template <bool SEGMENTS>
__global__ void __launch_bounds__(kBlock) k_pool_rows(int64_t n, int per_wave, const int64_t* __restrict__ offsets,
                                                      const int64_t* __restrict__ starts, Pool pool,
                                                      int64_t capacity, int64_t* __restrict__ ii, int64_t* __restrict__ jj,
                                                      double4* __restrict__ xy) {
  const int lane = lane_id();
  const int64_t q0 = ((int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * per_wave;
  const int64_t q = q0 + lane;
  long long o = 0, s = 0;
  int m = 0;
  if (lane < per_wave && q < n) {
    o = offsets[q];
    s = starts[q];
    const long long end = offsets[q + 1];
    if (s >= 0 && end <= capacity) m = (int)(end - o);
  }
  int incl = m;
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  const int excl = incl - m;
  const int total = __shfl(incl, 63);
  o -= excl;  // row g of the wavefront's rows is output row o + g of its owner,
  s -= excl;  // from pool entry s + g
  for (int base = 0; base < total; base += 64 * kAhead) {
    int own[kAhead], g[kAhead];  // g: past the end, the last row again (not stored)
    long long r[kAhead], from[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      own[u] = 0;
      g[u] = min(base + u * 64 + lane, total - 1);
    }
    for (int step = 32; step > 0; step >>= 1) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int e = __shfl(excl, own[u] + step);
        if (e <= g[u]) own[u] += step;
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      r[u] = __shfl(o, own[u]) + g[u];
      from[u] = __shfl(s, own[u]) + g[u];
    }
    if constexpr (SEGMENTS) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u) from[u] = pool.src[from[u]];
    }
    int c[kAhead];
    double4 v[SEGMENTS ? kAhead : 1];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      c[u] = pool.cell[from[u]];
      if constexpr (SEGMENTS) v[u] = pool.xy[from[u]];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (base + u * 64 + lane < total) {
        ii[r[u]] = q0 + own[u];
        jj[r[u]] = c[u];
        if constexpr (SEGMENTS) xy[r[u]] = v[u];
      }
    }
  }
}

struct GatherArgs {
  const ct_tree* tree;
  const double* qs;
  const int32_t* order;
  int64_t n;
  Pool pool;
  GatherParams p;
  int64_t* counts;
  int64_t* starts;
  int64_t* tail;
  hipStream_t st;
  template <int KIND, int MAXV>
  int run() const {
    k_gather<KIND, MAXV><<<gather_grid((n + p.per_wave - 1) / p.per_wave), 64, p.stack * sizeof(uint32_t), st>>>(
        view(tree), qs, order, n, p, pool, counts, starts, tail);
    CT_LAUNCH_CHECK();
    return CT_OK;
  }
  int go(int kind) const {
    const int nm = tree->n_max_vert;
    if (kind == kBoxes) return run<kBoxes, 4>();
    if (kind == kEdges) return run<kEdges, 4>();
    if (nm <= 4) return run<kFaces, 4>();
    if (nm <= 8) return run<kFaces, 8>();
    if (nm <= 16) return run<kFaces, 16>();
    return run<kFaces, 32>();
  }
};

}  // namespace

int launch_pool_rows(bool segments, int64_t n, const int64_t* offsets, const int64_t* starts, const int32_t* pool_cell,
                     const double* pool_xy, const int32_t* pool_src, int64_t capacity, int64_t* ii, int64_t* jj,
                     double* xy, hipStream_t st) {
  const Pool pool{const_cast<int32_t*>(pool_cell), reinterpret_cast<double4*>(const_cast<double*>(pool_xy)),
                  const_cast<int32_t*>(pool_src), 0, 1, 0};
  int per_wave = 64;
  while (per_wave > 1 && n < (int64_t)per_wave * kRowWaves) per_wave >>= 1;
  const int64_t per_block = (int64_t)per_wave * (kBlock / 64);
  const unsigned grid = (unsigned)((n + per_block - 1) / per_block);
  if (segments)
    k_pool_rows<true><<<grid, kBlock, 0, st>>>(n, per_wave, offsets, starts, pool, capacity, ii, jj, reinterpret_cast<double4*>(xy));
  else
    k_pool_rows<false><<<grid, kBlock, 0, st>>>(n, per_wave, offsets, starts, pool, capacity, ii, jj, nullptr);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // namespace ct

using namespace ct;

extern "C" {

int64_t ct_gather_tail_words(void) { return kTailWords; }

int64_t ct_gather_pool_rows(int32_t kind, int64_t n) {
  if (n <= 0) return 0;
  // Boxes (4 bytes a row): every list full, and as much for the boxes of ct_long.hip.  Segments (40 bytes): what
  // a group takes (half more rows than expected) if every list is full, as far as 2^26 rows go, and of
  // more than a million segments 64 each.
  if (kind == kBoxes) return (int64_t)2 * kBoxHits * n;
  return std::max((int64_t)64 * n, std::min((int64_t)384 * n, (int64_t)1 << 26));
}

int ct_gather_count(const ct_tree* tree, int32_t kind, const double* queries, int64_t n, const int32_t* order,
                    const int32_t* visit_cells, int64_t pool_rows, int32_t* pool_cell, double* pool_xy,
                    int32_t* pool_src, int64_t* counts, int64_t* starts, int64_t* tail, void* stream) {
  int rc = check_gather(tree, kind, n);
  if (rc) return rc;
  CT_REQUIRE(tail != nullptr && (n == 0 || (queries && counts && starts)), "null pointer");
  CT_REQUIRE(kind != kBoxes || visit_cells, "box queries need the cells by visit number");
  CT_REQUIRE(pool_rows >= 0 && pool_rows < ((int64_t)1 << 31) &&
                 (pool_rows == 0 || (pool_cell && (kind == kBoxes || (pool_xy && pool_src)))),
             "bad pool");
  hipStream_t st = as_stream(stream);
  rc = fill<int64_t>(tail, kTailWords, 0, st);
  if (rc || n == 0) return rc;
  GatherArgs a{};
  a.tree = tree;
  a.qs = queries;
  a.order = order;
  a.n = n;
  a.p = gather_params(tree, n, visit_cells, kind);
  a.pool = gather_pool(pool_rows, n, a.p.per_wave, pool_cell, pool_xy, pool_src);
  a.counts = counts;
  a.starts = starts;
  a.tail = tail;
  a.st = st;
  return a.go(kind);
}

int ct_gather_rows(int32_t kind, int64_t n, const int64_t* offsets, const int64_t* starts, const int32_t* pool_cell,
                   const double* pool_xy, const int32_t* pool_src, int64_t* ii, int64_t* jj, double* xy, void* stream) {
  CT_REQUIRE(kind >= kBoxes && kind <= kEdges && n >= 0 && (n == 0 || (offsets && starts)), "bad arguments");
  if (n == 0) return CT_OK;
  return launch_pool_rows(kind != kBoxes, n, offsets, starts, pool_cell, pool_xy, pool_src, INT64_MAX, ii, jj, xy,
                          as_stream(stream));
}

int ct_gather_left(int64_t n, const int64_t* starts, int64_t n_left, int32_t* left, int64_t* found, void* stream) {
  CT_REQUIRE(n >= 0 && n < ((int64_t)1 << 31) && n_left >= 0 && found && (n == 0 || starts) && (n_left == 0 || left),
             "bad arguments");
  hipStream_t st = as_stream(stream);
  const int rc = fill<int64_t>(found, 1, 0, st);
  if (rc || n == 0) return rc;
  k_left<<<grid_for(n), kBlock, 0, st>>>(n, starts, left, n_left, reinterpret_cast<unsigned long long*>(found));
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // extern "C"
