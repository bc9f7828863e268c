// ct_gather.hip -- box and segment queries, one wavefront for a few queries.
//
// A walk with one lane per query (query.py:177-244, 357-455) leaves four fifths of a wavefront idle
// (counted: 19 % of the VALU lanes active in the walks of 1e6 boxes and of 1e6 segments): the walks
// differ in length, and lanes wait for each other at every leaf.  Here the wavefront shares its
// queries' work: an LDS stack of (node, query) entries, of which every step takes the top 64, one
// per lane, and pushes their viable children; leaves put their cells on a second list, tested 64 at a
// time; segments put the cells whose box test passes on a third, clipped 64 at a time.  Every
// lane works at every step, whoever's query it is.
//
// The reference's row order is restored at the end.  A depth-first walk that enters the right
// child first visits the leaves by descending position in bb_indices and a leaf's cells by
// ascending position, so the cell at position k of leaf [ptr, ptr + size) is the walk's
// (n - ptr - size + k - ptr)-th: its visit number.  A query's box hits sorted by visit number are
// the reference's rows (a bitonic sort of (query, visit number) words in registers), and its
// segment hits are ranked by t, ties by visit number, as a stable sort by t ranks them.
//
// What bounds it: the latency of a step's loads (a node record, a cell box, a clip's vertices), hidden by
// the 15 to 20 wavefronts a CU holds (LDS, registers); the FP64 arithmetic of the segment tests is
// about half of the segments' time.  1e6 queries on a million-cell mesh, before (subqueries, one lane
// each, and their replay and sort kernels) and now, whole calls: boxes (31.6e6 rows) 1.94 and 1.22 ms,
// segments (13.6e6 rows) 3.50 and 2.50 ms; 2e3 segments 560 and 119 us.
//
// Rows go to a pool (each wavefront allocates from one of several counters); an exclusive scan of
// the counts gives the output offsets, and the copy kernels write whole output lines in query order.
// A query with more hits than the LDS lists hold, or that the pool has no room for, is left to the
// caller (starts[q] = -1): the subquery path (ct_split.hip) takes it.
#include <algorithm>
#include <cmath>

#include "ct_internal.h"
#include "ct_primitives.h"
#include "ct_traverse.h"

namespace ct {
namespace {

using Key = unsigned long long;

constexpr int kBoxes = 1, kFaces = 2, kEdges = 3;

// Queries of a wavefront's block of positions.
constexpr int kMaxPerWave = 16;

// Words of the lists: the owner (query of the block) above an index or visit number.  Trees of
// 2^26 cells or nodes and more are not taken (kMaxRecords).
constexpr int kOwnerShift = 27;
constexpr uint32_t kIndexMask = (1u << kOwnerShift) - 1u;
constexpr int64_t kMaxRecords = (int64_t)1 << 26;

// LDS list lengths.  The stack: a step of P entries needs room for P more; P shrinks as the stack
// fills, and depth + 1 places always remain for a single entry's way down (kStack + depth + 1 in all).
constexpr int kStack = 512;
constexpr int kCells = 192;  // 63 left over + 2 per lane
constexpr int kCands = 128;  // 63 left over + 64
// Hits a wavefront holds, and the expected hits of the queries it walks together: fewer and the steps
// at either end of a walk (few entries on the stack) weigh more, more and LDS limits the wavefronts in
// flight or groups overflow and are walked again one by one.  Measured, 1e6 queries, milliseconds:
// boxes 768/384 1.27, 768/480 1.22, 768/576 1.27, 512/384 1.91, 640/640 1.59;
// segments 256/160 2.67, 256/224 2.55, 320/280 2.50, 384/336 2.65, 512/448 2.77.
constexpr int kBoxHits = 768, kBoxGroup = 480;
constexpr int kSegHits = 320, kSegGroup = 280;

// Counters for pool allocation, each on its own 128-byte line: one counter for all wavefronts
// would serialize them (about 11 ns per atomic on one address).
constexpr int kPools = 64, kCounterStride = 16;
constexpr int kRowChunk = 512;  // pool rows a wavefront takes at a time (segments)

// Per-call words behind the offsets: [0] queries left to the caller, then the pool counters.
constexpr int kTailWords = 1 + kPools * kCounterStride;

struct Pool {
  int32_t* cell;   // boxes: the rows; segments: the hit cells
  double4* xy;     // segments: clipped pieces
  int32_t* src;    // segments: rows in output order -> entry of cell / xy
  int64_t rows;    // per counter
  int counters;
};

struct GatherParams {
  const int32_t* visit;  // boxes: the cell of every visit number
  double cell;           // typical cell side
  double reach;          // largest coordinate magnitude of the tree's bbox
  int per_wave;          // positions per wavefront
  int group;             // expected hits of the queries walked together
  int stack;             // stack entries
  int depth1;            // tree depth + 1
};

// Query data in LDS, by owner.
struct BoxRec {
  double4 d;
};

struct SegRec {
  double4 d;                  // (a, b)
  // for the node-box test (seg_near)
  double sx0, sx1, sy0, sy1;  // the segment's box, grown
  double ax2, ay2, dx, dy;    // 2 a, b - a
  double mm;
  int prune;                  // 1: node boxes decide; 0: query.py:407-441's tests (seg_children)
  int pad;
};

template <int KIND>
struct RecOf {
  using type = SegRec;
};
template <>
struct RecOf<kBoxes> {
  using type = BoxRec;
};
template <int KIND>
using QueryRec = typename RecOf<KIND>::type;

// Whether a segment comes near a node box: the separating axes x, y and the segment's normal, the
// box grown by m = 1e-9 * (largest coordinate magnitude of the segment and the tree).  Why a box that
// fails holds no hit: seg_meets_box (ct_traverse.h), with the larger of its margins; one cross product
// instead of two slab intersections (18 operations instead of 40).  NaN boxes pass.
__device__ __forceinline__ bool seg_near(const SegRec& r, double4 nb) {
  const bool off = nb.y < r.sx0 || nb.x > r.sx1 || nb.w < r.sy0 || nb.z > r.sy1;
  const double s = r.dx * ((nb.z + nb.w) - r.ay2) - r.dy * ((nb.x + nb.y) - r.ax2);
  const double reach = fabs(r.dx) * (nb.w - nb.z) + fabs(r.dy) * (nb.y - nb.x) + r.mm;
  return !(off || fabs(s) > reach);
}

// The slab test of the split dimension (query.py:228-242, 407-441; the t-tests of a segment that is
// not finite included).
template <int KIND>
__device__ __forceinline__ void slab(const QueryRec<KIND>& r, const NodeLd& nd, bool* left, bool* right) {
  if constexpr (KIND == kBoxes) {
    *left = (nd.dim ? r.d.z : r.d.x) <= nd.Lmax;
    *right = (nd.dim ? r.d.w : r.d.y) >= nd.Rmin;
  } else {
    SegPrune sp;
    sp.nbox = nullptr;
    sp.mseg = sp.ix = sp.iy = 0.0;
    sp.finite_v = isfinite(r.dx) && isfinite(r.dy);
    seg_children(nd, {r.d.x, r.d.y}, {r.d.z, r.d.w}, r.dx, r.dy, sp, left, right);
  }
}

// Bits of mask below this lane.
__device__ __forceinline__ int below(uint64_t mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// Record x of an array of 32-byte records (or its second half), through a 32-bit offset: the trees
// taken here have fewer than 2^26 nodes and cells.
template <typename T>
__device__ __forceinline__ T ld_rec(const void* __restrict__ base, uint32_t x, uint32_t half = 0) {
  return *reinterpret_cast<const T*>(static_cast<const char*>(base) + (x * 32u + half * 16u));
}

// Ascending bitonic sort of 64 * R words, word r * 64 + lane in v[r] of the lane.
template <int R>
__device__ __forceinline__ void wave_sort(uint32_t (&v)[R], int lane) {
#pragma unroll
  for (int k = 2; k <= 64 * R; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j >= 64) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int p = r ^ (j >> 6);
          if (p > r) {
            const bool up = ((r << 6) & k) == 0;
            const uint32_t a = v[r], b = v[p];
            v[r] = up ? min(a, b) : max(a, b);
            v[p] = up ? max(a, b) : min(a, b);
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const uint32_t o = __shfl_xor(v[r], j, 64);
          const bool low = ((((r << 6) | lane) & k) == 0) == ((lane & j) == 0);  // this lane keeps the smaller
          v[r] = (o < v[r]) == low ? o : v[r];
        }
      }
    }
  }
}

// The cells of the visit numbers in list[0, m), m <= 64 * R, in ascending order, to out.
template <int R>
__device__ __forceinline__ void sorted_cells(const uint32_t* list, int m, int lane,
                                             const int32_t* __restrict__ visit, int32_t* __restrict__ out) {
  uint32_t v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = r * 64 + lane < m ? list[r * 64 + lane] : ~0u;
  wave_sort<R>(v, lane);
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r * 64 + lane < m) out[r * 64 + lane] = visit[v[r] & kIndexMask];
}

// The lists hits (and ts, byown for segments), m <= 64 * R entries, grouped by owner: entry i to
// first[owner] + its arrival among the owner's.  byown: the entry's old place.
template <int R, bool SEGMENTS>
__device__ __forceinline__ void group_by_owner(uint32_t* hits, unsigned long long* ts, uint16_t* byown, int m, int lane,
                                               const int* first, int* cnt) {
  uint32_t w[R];
  unsigned long long t[SEGMENTS ? R : 1];
  int to[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = r * 64 + lane;
    to[r] = -1;
    if (i < m) {
      w[r] = hits[i];
      if constexpr (SEGMENTS) t[r] = ts[i];
      const int o = (int)(w[r] >> kOwnerShift);
      to[r] = first[o] + atomicSub(&cnt[o], 1) - 1;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (to[r] < 0) continue;
    hits[to[r]] = w[r];
    if constexpr (SEGMENTS) {
      ts[to[r]] = t[r];
      byown[to[r]] = (uint16_t)(r * 64 + lane);
    }
  }
  __syncthreads();
}

// row_t as a key whose unsigned order is np.lexsort's: -0.0 as 0.0, NaN last.
__device__ __forceinline__ unsigned long long t_key(double t) {
  return isnan(t) ? ~0ull : dkey(t + 0.0);
}

// Expected hits of a query (NaN and infinite ones: one).
template <int KIND>
__device__ __forceinline__ int expected(const QueryRec<KIND>& r, double cell) {
  double e;
  if constexpr (KIND == kBoxes) e = ((r.d.y - r.d.x) / cell + 1.0) * ((r.d.w - r.d.z) / cell + 1.0);
  else e = 1.5 * sqrt(r.dx * r.dx + r.dy * r.dy) / cell + 1.0;
  return e > 1.0 ? (e < 1e6 ? (int)e : 1000000) : 1;
}

// Whether a listed cell goes on: a box's whole test; a segment-edge pair's whole test; for a segment
// and a face what is cheap and rejects nearly all that Cohen-Sutherland rejects (its trivial
// rejection and seg_near): the exact test runs with the clip, where its loop diverges less.
template <int KIND>
__device__ __forceinline__ bool cell_test(const TreeView& t, const QueryRec<KIND>& r, int k, int* c, P2* cc, P2* dd) {
  const P2 a = {r.d.x, r.d.y}, b = {r.d.z, r.d.w};
  if constexpr (KIND == kEdges) {
    *c = t.bb_indices[k];
    return edge_edge(t, *c, a, b, cc, dd);
  } else {
    const double4 b4 = t.lbb ? ld_rec<double4>(t.lbb, (uint32_t)k) : ld_rec<double4>(t.bb, (uint32_t)t.bb_indices[k]);
    const Box bb{b4.x, b4.y, b4.z, b4.w};
    if constexpr (KIND == kBoxes) {
      return boxes_intersect(Box{r.d.x, r.d.y, r.d.z, r.d.w}, bb);
    } else {
      if ((cs_code(a, bb) & cs_code(b, bb)) != 0) return false;
      return r.prune == 0 || seg_near(r, make_double4(bb.xmin, bb.xmax, bb.ymin, bb.ymax));
    }
  }
}

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

// counts[q], starts[q] (the query's first pool row; -1: left to the caller) and the pool's rows.
// One wavefront per workgroup: its LDS is its own, and the hardware's workgroup scheduler balances
// the blocks.
template <int KIND, int MAXV>
__global__ void __launch_bounds__(64, MAXV <= 8 ? 4 : 1)
k_gather(TreeView t, const double* __restrict__ qs, const int32_t* __restrict__ order, int64_t n, GatherParams p,
         Pool pool, int64_t* __restrict__ counts, int64_t* __restrict__ starts, int64_t* tail) {
  constexpr int kHits = KIND == kBoxes ? kBoxHits : kSegHits;
  extern __shared__ uint32_t stack[];  // p.stack entries
  __shared__ QueryRec<KIND> recs[kMaxPerWave];
  __shared__ uint2 cells[kCells];                         // (owner | position, owner | visit number)
  __shared__ uint2 cands[KIND == kFaces ? kCands : 1];    // segment-face: box test passed
  __shared__ uint32_t hits[kHits];                        // owner | visit number
  __shared__ Key ts[KIND == kBoxes ? 1 : kHits];           // segments: t_key
  __shared__ uint16_t byown[KIND == kBoxes ? 1 : kHits];   // segments: a grouped hit's pool row
  __shared__ int cnt[kMaxPerWave], first[kMaxPerWave + 1];
  const int lane = lane_id();
  const int64_t i0 = block_of(blockIdx.x) * p.per_wave;
  if (i0 >= n) return;
  const int nq = (int)min((int64_t)p.per_wave, n - i0);

  // Each lane one query: down from the root while a single child is viable.
  int64_t q = 0;
  int start = -1, weight = 0;
  if (lane < nq) {
    q = query_index(order, i0 + lane);
    QueryRec<KIND> rec;
    rec.d = reinterpret_cast<const double4*>(qs)[q];
    bool in;
    if constexpr (KIND == kBoxes) {
      in = boxes_intersect(Box{rec.d.x, rec.d.y, rec.d.z, rec.d.w}, t.bbox);
    } else {
      const P2 a = {rec.d.x, rec.d.y}, b = {rec.d.z, rec.d.w};
      rec.dx = b.x - a.x;
      rec.dy = b.y - a.y;
      rec.ax2 = 2.0 * a.x;
      rec.ay2 = 2.0 * a.y;
      const double mseg = pmax(pmax(fabs(a.x), fabs(a.y)), pmax(fabs(b.x), fabs(b.y)));
      const double m = 1e-9 * pmax(mseg, p.reach);
      rec.sx0 = pmin(a.x, b.x) - m;
      rec.sx1 = pmax(a.x, b.x) + m;
      rec.sy0 = pmin(a.y, b.y) - m;
      rec.sy1 = pmax(a.y, b.y) + m;
      rec.mm = 2.0 * m * (fabs(rec.dx) + fabs(rec.dy));
      rec.prune = KIND == kFaces && t.nbox != nullptr && isfinite(mseg) && isfinite(rec.mm) && isfinite(rec.dx) &&
                  isfinite(rec.dy);
      P2 c0, d0;
      in = cohen_sutherland(a, b, t.bbox, &c0, &d0);
    }
    if (in) {
      weight = expected<KIND>(rec, p.cell);
      start = 0;
      while (true) {
        const NodeLd nd = ld_node(t.nodes, start);
        if (nd.child == -1) break;
        bool left, right;
        slab<KIND>(rec, nd, &left, &right);
        if (left && right) break;
        if (!left && !right) {
          start = -1;
          break;
        }
        start = nd.child + (right ? 1 : 0);
      }
    }
    recs[lane] = rec;
  }

  const int sub = (int)(blockIdx.x % (unsigned)pool.counters);
  unsigned long long* ctr = reinterpret_cast<unsigned long long*>(tail) + 1 + sub * kCounterStride;
  const long long pool0 = (long long)sub * pool.rows;
  long long row_at = 0, row_end = 0;  // segments: the wavefront's pool rows
  int single_until = 0;               // queries before this one are walked alone
  for (int g0 = 0; g0 < nq;) {
    // The next queries whose expected hits fill a list (at least one).
    int g1 = g0 + 1;
    int x = lane >= g0 && lane < nq && start >= 0 ? weight : 0;
    for (int d = 1; d < kMaxPerWave; d <<= 1) {
      const int y = __shfl_up(x, d);
      if (lane >= d) x += y;
    }
    if (g0 >= single_until) {
      const uint64_t past = __ballot(lane > g0 && lane < nq && x > p.group);
      g1 = past ? __ffsll((unsigned long long)past) - 1 : nq;
    }
    const bool mine = lane >= g0 && lane < g1;
    const uint64_t alive = __ballot(mine && start >= 0);
    const int wsum = __shfl(x, g1 - 1);
    auto owner = [](uint32_t w) { return (int)(w >> kOwnerShift); };
    __syncthreads();  // one wavefront: orders LDS accesses
    if (lane < kMaxPerWave) cnt[lane] = 0;
    if (mine && start >= 0)
      stack[below(alive)] = (uint32_t)lane << kOwnerShift | (uint32_t)start;
    // Hits this group may have: the lists' length, and the pool rows at hand (segments).
    int room = kHits;
    if (KIND != kBoxes && alive) {
      const int want = g1 - g0 == 1 ? kHits : min(kHits, 2 * wsum + 32);
      if (row_end - row_at < want) {
        long long at = 0;
        if (lane == 0) at = (long long)atomicAdd(ctr, (unsigned long long)kRowChunk);
        at = __shfl(at, 0);
        row_at = pool0 + at;
        row_end = at + kRowChunk > pool.rows ? row_at : row_at + kRowChunk;
      }
      room = (int)min((long long)kHits, row_end - row_at);
    }
    __syncthreads();
    int sp = __popcll(alive), ncell = 0, ncand = 0, nhit = 0;
    bool over = false;  // more hits than `room`, or a leaf larger than the cell list
    while (true) {
      // a full list first: each step leaves room for what the next one adds
      if (KIND == kFaces && (ncand >= 64 || (sp == 0 && ncell == 0 && ncand > 0))) {
        const int take = min(64, ncand);
        ncand -= take;
        bool hit = lane < take;
        uint2 e = make_uint2(0u, 0u);
        P2 cc{}, dd{};
        int c = 0;
        double4 d{};
        if (hit) {
          e = cands[ncand + lane];
          const int k = (int)(e.x & kIndexMask);
          d = recs[owner(e.x)].d;
          c = t.bb_indices[k];
          const P2 a = {d.x, d.y}, b = {d.z, d.w};
          const Box bb = leaf_box(t, k, c);
          hit = cohen_sutherland(a, b, bb, &cc, &dd);
          if (hit) {
            if (t.leaf != nullptr) hit = edge_face_clip_row<MAXV>(t, k, c, a, b, &cc, &dd);
            else hit = edge_face_clip<MAXV>(t, c, bb, a, b, &cc, &dd);
          }
        }
        const uint64_t mask = __ballot(hit);
        const int got = __popcll(mask), at = nhit + below(mask);
        if (nhit + got > room) {
          over = true;
          break;
        }
        if (hit) {
          hits[at] = e.y;
          ts[at] = t_key(row_t(d, make_double2(cc.x, cc.y)));
          atomicAdd(&cnt[owner(e.y)], 1);
          pool.cell[row_at + at] = c;
          pool.xy[row_at + at] = make_double4(cc.x, cc.y, dd.x, dd.y);
        }
        nhit += got;
        __syncthreads();
        continue;
      }
      if (ncell >= 64 || (sp == 0 && ncell > 0)) {
        const int take = min(64, ncell);
        ncell -= take;
        bool hit = lane < take;
        uint2 e = make_uint2(0u, 0u);
        P2 cc{}, dd{};
        int c = 0;
        if (hit) {
          e = cells[ncell + lane];
          hit = cell_test<KIND>(t, recs[owner(e.x)], (int)(e.x & kIndexMask), &c, &cc, &dd);
        }
        const uint64_t mask = __ballot(hit);
        const int got = __popcll(mask), at = below(mask);
        if constexpr (KIND == kFaces) {
          if (hit) cands[ncand + at] = e;
          ncand += got;
        } else {
          if (nhit + got > room) {
            over = true;
            break;
          }
          if (hit) {
            hits[nhit + at] = e.y;
            atomicAdd(&cnt[owner(e.y)], 1);
            if constexpr (KIND == kEdges) {
              ts[nhit + at] = t_key(row_t(recs[owner(e.y)].d, make_double2(cc.x, cc.y)));
              pool.cell[row_at + nhit + at] = c;
              pool.xy[row_at + nhit + at] = make_double4(cc.x, cc.y, dd.x, dd.y);
            }
          }
          nhit += got;
        }
        __syncthreads();
        continue;
      }
      if (sp == 0) break;
      // the top of the stack
      const int take = min(min(64, sp), max(1, p.stack - p.depth1 - sp));
      sp -= take;
      bool left = false, right = false;
      uint32_t e = 0;
      int child = 0, ptr = 0, size = 0;
      if (lane < take) {
        e = stack[sp + lane];
        const uint32_t x = e & kIndexMask;
        const QueryRec<KIND>& r = recs[owner(e)];
        bool here = true, by_box = false;
        NodeLd nd;
        if constexpr (KIND == kFaces) by_box = r.prune != 0;
        if (by_box) {
          // A segment tests the node's own box, loaded beside its record: one round of loads a step
          // (testing the children's boxes before pushing them takes two, one after the other).
          // Every cell it can hit lies in the boxes it comes near, so the slab test adds nothing.
          if constexpr (KIND == kFaces) {
            const int4 w = ld_rec<int4>(t.nodes, x, 1);
            here = seg_near(r, ld_rec<double4>(t.nbox, x + 1));
            nd = NodeLd{0.0, 0.0, w.x, w.y, w.z, w.w};
          }
          left = right = here && nd.child != -1;
        } else {
          const double2 lr = ld_rec<double2>(t.nodes, x);
          const int4 w = ld_rec<int4>(t.nodes, x, 1);
          nd = NodeLd{lr.x, lr.y, w.x, w.y, w.z, w.w};
          if (nd.child != -1) slab<KIND>(r, nd, &left, &right);
        }
        child = nd.child;
        if (here && child == -1) {
          ptr = nd.ptr;
          size = nd.size;
        }
      }
      const uint32_t tag = e & ~kIndexMask;
      const uint32_t v0 = (uint32_t)(t.n_elements - ptr - size);
      __syncthreads();  // the popped entries are read
      const uint64_t ml = __ballot(left), mr = __ballot(right);
      if (left) stack[sp + below(ml)] = tag | (uint32_t)child;
      sp += __popcll(ml);
      if (right) stack[sp + below(mr)] = tag | (uint32_t)(child + 1);
      sp += __popcll(mr);
      // leaves: their cells (fewer than 64 are listed here, and 128 more fit)
      if (!__any(size > 2)) {
        const uint64_t m0 = __ballot(size > 0), m1 = __ballot(size > 1);
        if (size > 0) cells[ncell + below(m0)] = make_uint2(tag | (uint32_t)ptr, tag | v0);
        ncell += __popcll(m0);
        if (size > 1) cells[ncell + below(m1)] = make_uint2(tag | (uint32_t)(ptr + 1), tag | (v0 + 1));
        ncell += __popcll(m1);
      } else {
        // larger leaves: those that fit; the others go back to the stack
        int incl = size;
        for (int d = 1; d < 64; d <<= 1) {
          const int y = __shfl_up(incl, d);
          if (lane >= d) incl += y;
        }
        const bool fits = incl <= kCells - ncell;
        const uint64_t back = __ballot(size > 0 && !fits), put = __ballot(size > 0 && fits);
        if (back && !put) {  // a leaf larger than the list
          over = true;
          break;
        }
        if (size > 0 && fits)
          for (int j = 0; j < size; ++j)
            cells[ncell + incl - size + j] = make_uint2(tag | (uint32_t)(ptr + j), tag | (v0 + j));
        if (size > 0 && !fits) stack[sp + below(back)] = e;
        sp += __popcll(back);
        // the listed cells: the prefix of the last lane that fits
        const int last = 63 - __clzll((unsigned long long)put);
        ncell += put ? __shfl(incl, last) : 0;
      }
      __syncthreads();
    }

    bool left_over = over;  // the group's queries are left to the caller
    if (over && g1 - g0 > 1 && (KIND == kBoxes || room == kHits || row_end > row_at)) {
      single_until = g1;  // again, one query at a time
      continue;
    }
    // ranges of the owners' hits
    __syncthreads();
    const int c_own = mine && !over ? cnt[lane] : 0;
    int incl = c_own;
    for (int d = 1; d < kMaxPerWave; d <<= 1) {
      const int y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    const int my_first = incl - c_own;
    if (lane < kMaxPerWave) {
      first[lane] = my_first;
      if (lane == kMaxPerWave - 1) first[kMaxPerWave] = incl;
    }
    __syncthreads();
    long long at = row_at;
    if (!over && nhit > 0) {
      if constexpr (KIND == kBoxes) {
        if (lane == 0) at = (long long)atomicAdd(ctr, (unsigned long long)nhit);
        at = __shfl(at, 0);
        left_over = at + nhit > pool.rows;
        at += pool0;
        if (!left_over) {
          if (g1 - g0 > 1) {
            if (nhit <= 256) group_by_owner<4, false>(hits, nullptr, nullptr, nhit, lane, first, cnt);
            else group_by_owner<kBoxHits / 64, false>(hits, nullptr, nullptr, nhit, lane, first, cnt);
          }
          // as many owners at a time as 64 words hold, or one larger owner
          for (int o = g0; o < g1;) {
            const int f = __shfl(my_first, o);
            const uint64_t fit = __ballot(lane >= o && lane < g1 && incl - f <= 64) >> o;
            int e = o + (fit ? (~fit ? __ffsll((unsigned long long)~fit) - 1 : 64) : 0);
            e = max(e, o + 1);
            const int m = __shfl(incl, e - 1) - f;
            int32_t* const out = pool.cell + at + f;
            if (m <= 64) sorted_cells<1>(hits + f, m, lane, p.visit, out);
            else if (m <= 128) sorted_cells<2>(hits + f, m, lane, p.visit, out);
            else if (m <= 256) sorted_cells<4>(hits + f, m, lane, p.visit, out);
            else if (m <= 512) sorted_cells<8>(hits + f, m, lane, p.visit, out);
            else sorted_cells<16>(hits + f, m, lane, p.visit, out);
            o = e;
          }
        }
      } else {
        const bool grouped = g1 - g0 > 1;
        if (grouped) group_by_owner<kSegHits / 64, true>(hits, ts, byown, nhit, lane, first, cnt);
        // geometry_utils.py:564-574: by t (NaN last), then in the walk's order
        for (int s = lane; s < nhit; s += 64) {
          const uint32_t wi = hits[s];
          const Key ti = ts[s];
          const int o = owner(wi), f = first[o], l = first[o + 1];
          int r = f, same = 0;
          for (int k = f; k < l; ++k) {
            const Key tj = ts[k];
            r += tj < ti ? 1 : 0;
            same += tj == ti ? 1 : 0;
          }
          if (same > 1)
            for (int k = f; k < l; ++k) r += ts[k] == ti && hits[k] < wi ? 1 : 0;
          pool.src[at + r] = (int32_t)(at + (grouped ? byown[s] : s));
        }
        row_at += nhit;
      }
    }
    if (mine) {
      const bool leave = left_over && (over ? start >= 0 : c_own > 0);
      counts[q] = leave ? 0 : c_own;
      starts[q] = leave ? -1 : at + my_first;
      if (leave) atomicAdd(reinterpret_cast<unsigned long long*>(tail), 1ull);
    }
    g0 = g1;
  }
}

// Output rows from the pool, 64 queries per wavefront in query order: their rows are one run of
// the output, written 64 rows per step (row g's owner by a binary search over the wavefront's
// prefix), so every output line is written whole.  kAhead steps run together: a row is a chain of two
// or three loads.
constexpr int kAhead = 4;

template <bool SEGMENTS>
__global__ void __launch_bounds__(kBlock) k_pool_rows(int64_t n, const int64_t* __restrict__ offsets,
                                                      const int64_t* __restrict__ starts, Pool pool,
                                                      int64_t* __restrict__ ii, int64_t* __restrict__ jj,
                                                      double4* __restrict__ xy) {
  const int lane = lane_id();
  const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t q0 = q - lane;
  long long o = 0, s = 0;
  int m = 0;
  if (q < n) {
    o = offsets[q];
    s = starts[q];
    if (s >= 0) m = (int)(offsets[q + 1] - o);
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

// The rows of a batch of left-over queries (sub-query s of them is query idx[s]; its rows at
// sub_offsets[s]) to their places among all rows.
__global__ void __launch_bounds__(kBlock) k_place_rows(int64_t rows, const int64_t* __restrict__ idx,
                                                       const int64_t* __restrict__ sub_offsets,
                                                       const int64_t* __restrict__ offsets,
                                                       const int64_t* __restrict__ sub_ii,
                                                       const int64_t* __restrict__ sub_jj,
                                                       const double4* __restrict__ sub_xy, int64_t* __restrict__ ii,
                                                       int64_t* __restrict__ jj, double4* __restrict__ xy) {
  const int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (r >= rows) return;
  const int64_t s = sub_ii[r], q = idx[s], o = offsets[q] + (r - sub_offsets[s]);
  ii[o] = q;
  jj[o] = sub_jj[r];
  if (xy) xy[o] = sub_xy[r];
}

// The cell of every visit number.
__global__ void __launch_bounds__(kBlock) k_visit_cells(const ct_node* __restrict__ nodes, int64_t n_nodes,
                                                        const int32_t* __restrict__ bb_indices, int n,
                                                        int32_t* __restrict__ out) {
  const int64_t x = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (x >= n_nodes) return;
  const ct_node nd = nodes[x];
  if (nd.child != -1) return;
  for (int j = 0; j < nd.size; ++j) out[n - nd.ptr - nd.size + j] = bb_indices[nd.ptr + j];
}

GatherParams params(const ct_tree* tree, int64_t n, const int32_t* visit, int kind) {
  GatherParams p{};
  p.visit = visit;
  const double ex = tree->bbox[1] - tree->bbox[0], ey = tree->bbox[3] - tree->bbox[2];
  p.cell = sqrt(ex * ey / (double)tree->n_elements);
  if (!(p.cell > 0.0)) p.cell = 1.0;  // degenerate bbox (only how queries are grouped depends on it)
  for (double v : tree->bbox) p.reach = std::max(p.reach, std::fabs(v));
  // Few queries: fewer per wavefront, so that at least 4096 wavefronts share the work (256 CUs hold
  // about 4000 of them); many: 16 (8 per wavefront: 1e6 boxes 1.41 instead of 1.22
  // ms, 1e6 segments 2.74 instead of 2.67: too few entries on the stack to fill the lanes).
  p.per_wave = (int)std::min((int64_t)kMaxPerWave, std::max((int64_t)1, n / 4096));
  p.depth1 = tree->depth + 1;
  p.stack = kStack + p.depth1;
  p.group = kind == kBoxes ? kBoxGroup : kSegGroup;
  return p;
}

Pool make_pool(int64_t rows, int64_t n, int per_wave, int32_t* cell, double* xy, int32_t* src) {
  const int64_t waves = (n + per_wave - 1) / per_wave;
  Pool pool{cell, reinterpret_cast<double4*>(xy), src, 0, 1};
  pool.counters = (int)std::min((int64_t)kPools, std::max((int64_t)1, waves / 64));
  pool.rows = rows / pool.counters;
  return pool;
}

int check_gather(const ct_tree* tree, int32_t kind, int64_t n) {
  CT_REQUIRE(tree != nullptr && tree->nodes && tree->bb_indices && tree->elements && tree->vertices && tree->bb_coords,
             "incomplete tree");
  CT_REQUIRE(tree->depth >= 0 && tree->depth <= CT_MAX_DEPTH, "trees of depth <= %d", CT_MAX_DEPTH);
  CT_REQUIRE(tree->n_nodes < kMaxRecords && tree->n_elements < kMaxRecords, "trees of fewer than 2^26 nodes and cells");
  CT_REQUIRE(kind >= kBoxes && kind <= kEdges, "kind must be 1 (boxes), 2 (segment-face) or 3 (segment-edge)");
  CT_REQUIRE(kind == kEdges ? tree->n_max_vert == 2 : (kind == kBoxes || tree->n_max_vert >= 3),
             "kind does not match the tree");
  CT_REQUIRE(n >= 0 && n < ((int64_t)1 << 31), "n must be in [0, 2^31)");
  return CT_OK;
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
}  // namespace ct

using namespace ct;

extern "C" {

int64_t ct_gather_tail_words(void) { return kTailWords; }

int64_t ct_gather_pool_rows(int32_t kind, int64_t n) {
  if (n <= 0) return 0;
  // boxes: 256 hits per query; segments: 64 per query, at least a chunk per wavefront
  if (kind == kBoxes) return std::max((int64_t)256 * n, (int64_t)kBoxHits);
  const int64_t per_wave = std::min((int64_t)kMaxPerWave, std::max((int64_t)1, n / 4096));
  return std::max((int64_t)64 * n, ((n + per_wave - 1) / per_wave * 5 / 4 + kPools) * kRowChunk);
}

int ct_visit_cells(const ct_tree* tree, int32_t* out, void* stream) {
  CT_REQUIRE(tree && tree->nodes && tree->bb_indices && out, "bad arguments");
  k_visit_cells<<<grid_for(tree->n_nodes), kBlock, 0, as_stream(stream)>>>(tree->nodes, tree->n_nodes, tree->bb_indices,
                                                                         (int)tree->n_elements, out);
  CT_LAUNCH_CHECK();
  return CT_OK;
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
  a.p = params(tree, n, visit_cells, kind);
  a.pool = make_pool(pool_rows, n, a.p.per_wave, pool_cell, pool_xy, pool_src);
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
  const Pool pool{const_cast<int32_t*>(pool_cell), reinterpret_cast<double4*>(const_cast<double*>(pool_xy)),
                  const_cast<int32_t*>(pool_src), 0, 1};
  hipStream_t st = as_stream(stream);
  if (kind == kBoxes) k_pool_rows<false><<<grid_for(n), kBlock, 0, st>>>(n, offsets, starts, pool, ii, jj, nullptr);
  else k_pool_rows<true><<<grid_for(n), kBlock, 0, st>>>(n, offsets, starts, pool, ii, jj, reinterpret_cast<double4*>(xy));
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_place_rows(int64_t rows, const int64_t* idx, const int64_t* sub_offsets, const int64_t* offsets,
                  const int64_t* sub_ii, const int64_t* sub_jj, const double* sub_xy, int64_t* ii, int64_t* jj,
                  double* xy, void* stream) {
  CT_REQUIRE(rows >= 0 && (rows == 0 || (idx && sub_offsets && offsets && sub_ii && sub_jj && ii && jj)), "bad arguments");
  CT_REQUIRE((sub_xy == nullptr) == (xy == nullptr), "sub_xy and xy go together");
  if (rows == 0) return CT_OK;
  k_place_rows<<<grid_for(rows), kBlock, 0, as_stream(stream)>>>(rows, idx, sub_offsets, offsets, sub_ii, sub_jj,
                                                               reinterpret_cast<const double4*>(sub_xy), ii, jj,
                                                               reinterpret_cast<double4*>(xy));
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // extern "C"
