// ct_gather.h -- walks of box and segment queries, one wavefront for a few queries.
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
#ifndef CT_GATHER_H
#define CT_GATHER_H

#include <algorithm>

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
constexpr int kStack = 240;
constexpr int kCells = 192;  // 63 left over + 2 per lane
constexpr int kCands = 128;  // 63 left over + 64
// A step with a leaf of more cells than this lists one leaf, 64 cells at a time by all lanes, and puts
// the others back: each lane listing its own leaf takes as many stores as the largest has cells, and a
// leaf may be larger than the list.  200,000 triangles in leaves of up to 130 cells, 1e5 boxes: 514 us,
// 771 lane by lane; of up to 64 cells, 1e5 segments: 857 lane by lane, 982 one leaf at a time.
constexpr int kLeafCells = 64;
// Hits a wavefront holds, and the expected hits of the queries it walks together: fewer and the steps
// at either end of a walk (few entries on the stack) weigh more, more and LDS limits the wavefronts in
// flight or groups overflow and are walked again one by one.  Measured, 1e6 queries, milliseconds:
// boxes 768/384 1.27, 768/480 1.22, 768/576 1.27, 512/384 1.91, 640/640 1.59;
// segments 256/160 2.67, 256/224 2.55, 320/280 2.50, 384/336 2.65, 512/448 2.77.  With 310/270 and the
// stack above, a segment wavefront's LDS is 10,240 bytes up to a depth of 43, and 16 of them fit a CU
// instead of 15: 2.55 -> 2.41.
// A box walked alone may have kBoxHits: boxes of 20 cell widths have 900 (8e3 of them on 20,000
// triangles: 0.16 ms, and 0.60 with 768).
constexpr int kBoxHits = 1024, kBoxGroupHits = 768, kBoxGroup = 480;
constexpr int kSegHits = 310, kSegGroup = 270;
// Counters for pool allocation, each on its own 128-byte line: one counter for all wavefronts
// would serialize them (about 11 ns per atomic on one address).
constexpr int kPools = 64, kCounterStride = 16;

// Per-call words behind the offsets: [0] queries left to the caller, then the pool counters.
constexpr int kTailWords = 1 + kPools * kCounterStride;

struct Pool {
  int32_t* cell;   // boxes: the rows; segments: the hit cells
  double4* xy;     // segments: clipped pieces
  int32_t* src;    // segments: rows in output order -> entry of cell / xy
  int64_t rows;    // per counter
  int counters;
  int chunk;       // segments: rows a wavefront takes at a time, at least (0: those it asks for)
};

// A wavefront's pool rows at hand (segments) and the counter it allocates from.
struct PoolRows {
  long long at = 0, end = 0;
  int sub;
  int tried = 0;  // counters found empty
  __device__ __forceinline__ unsigned long long* counter(int64_t* tail) const {
    return reinterpret_cast<unsigned long long*>(tail) + 1 + sub * kCounterStride;
  }
  // `want` rows or a chunk: from this wavefront's counter, or from the next that has them.
  __device__ __forceinline__ void refill(const Pool& pool, int64_t* tail, int want) {
    const int take = max(want, pool.chunk);
    at = end = 0;
    while (tried < pool.counters) {
      long long x = 0;
      if (lane_id() == 0) x = (long long)atomicAdd(counter(tail), (unsigned long long)take);
      x = __shfl(x, 0);
      if (x + take <= pool.rows) {
        at = (long long)sub * pool.rows + x;
        end = at + take;
        return;
      }
      sub = sub + 1 == pool.counters ? 0 : sub + 1;
      ++tried;
    }
  }
};

struct GatherParams {
  const int32_t* visit;  // boxes: the cell of every visit number
  double cell;           // typical cell side
  double reach;          // largest coordinate magnitude of the tree's bbox
  int per_wave;          // positions per wavefront
  int group;             // expected hits of the queries walked together
  int leave;             // expected hits beyond which a query is left without a walk likely in vain
  int stack;             // stack entries
  int depth1;            // tree depth + 1

  __host__ __device__ __forceinline__ void scale(const TreeView& t) {
    const double ex = t.bbox.xmax - t.bbox.xmin, ey = t.bbox.ymax - t.bbox.ymin;
    cell = sqrt(ex * ey / (double)t.n_elements);
    if (!(cell > 0.0)) cell = 1.0;  // degenerate bbox (only how queries are grouped depends on it)
    reach = fmax(fmax(fabs(t.bbox.xmin), fabs(t.bbox.xmax)), fmax(fabs(t.bbox.ymin), fabs(t.bbox.ymax)));
  }
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

// Query q's record; whether it meets the tree's bbox.
template <int KIND>
__device__ __forceinline__ bool load_query(const TreeView& t, const double* __restrict__ qs, int64_t q, double reach,
                                           QueryRec<KIND>* rec) {
  rec->d = reinterpret_cast<const double4*>(qs)[q];
  if constexpr (KIND == kBoxes) {
    return boxes_intersect(Box{rec->d.x, rec->d.y, rec->d.z, rec->d.w}, t.bbox);
  } else {
    const P2 a = {rec->d.x, rec->d.y}, b = {rec->d.z, rec->d.w};
    rec->dx = b.x - a.x;
    rec->dy = b.y - a.y;
    rec->ax2 = 2.0 * a.x;
    rec->ay2 = 2.0 * a.y;
    const double mseg = pmax(pmax(fabs(a.x), fabs(a.y)), pmax(fabs(b.x), fabs(b.y)));
    const double m = 1e-9 * pmax(mseg, reach);
    rec->sx0 = pmin(a.x, b.x) - m;
    rec->sx1 = pmax(a.x, b.x) + m;
    rec->sy0 = pmin(a.y, b.y) - m;
    rec->sy1 = pmax(a.y, b.y) + m;
    rec->mm = 2.0 * m * (fabs(rec->dx) + fabs(rec->dy));
    rec->prune = KIND == kFaces && t.nbox != nullptr && isfinite(mseg) && isfinite(rec->mm) && isfinite(rec->dx) &&
                 isfinite(rec->dy);
    P2 c0, d0;
    return cohen_sutherland<true>(a, b, t.bbox, &c0, &d0);
  }
}

// Down from the root while a single child is viable; -1: none is.
template <int KIND>
__device__ __forceinline__ int first_fork(const TreeView& t, const QueryRec<KIND>& rec) {
  int node = 0;
  while (true) {
    const NodeLd nd = ld_node(t.nodes, node);
    if (nd.child == -1) return node;
    bool left, right;
    slab<KIND>(rec, nd, &left, &right);
    if (left && right) return node;
    if (!left && !right) return -1;
    node = nd.child + (right ? 1 : 0);
  }
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

// counts[q], starts[q] (the query's first pool row; -1: left to the caller) and the pool's rows of
// the queries at positions [i0, i0 + nq), nq <= kMaxPerWave.  For workgroups of one wavefront:
// its LDS is its own, and the barriers only order its accesses.
template <int KIND, int MAXV>
__device__ __forceinline__ void gather_block(const TreeView& t, const double* __restrict__ qs,
                                             const int32_t* __restrict__ order, int64_t i0, int nq,
                                             const GatherParams& p, const Pool& pool, PoolRows& rows,
                                             int64_t* __restrict__ counts, int64_t* __restrict__ starts,
                                             int64_t* tail) {
  constexpr int kHits = KIND == kBoxes ? kBoxHits : kSegHits;
  extern __shared__ uint32_t stack[];  // p.stack entries
  __shared__ QueryRec<KIND> recs[kMaxPerWave];
  __shared__ uint2 cells[kCells];                         // (owner | position, owner | visit number)
  __shared__ uint2 cands[KIND == kFaces ? kCands : 1];    // segment-face: box test passed
  __shared__ uint32_t hits[kHits];                        // owner | visit number
  __shared__ Key ts[KIND == kBoxes ? 1 : kHits];           // segments: t_key
  __shared__ uint16_t byown[KIND == kBoxes ? 1 : kHits];   // segments: a grouped hit's pool row
  __shared__ int cnt[kMaxPerWave], first[kMaxPerWave + 1];
  __shared__ uint32_t leaf_done;                           // cells listed of the large leaf on top of the stack
  const int lane = lane_id();
  __syncthreads();  // one wavefront: the last block's LDS reads are over

  // Each lane one query: down from the root while a single child is viable.
  int64_t q = 0;
  int start = -1, weight = 0;
  bool big = false;
  if (lane < nq) {
    q = query_index(order, i0 + lane);
    QueryRec<KIND> rec;
    if (load_query<KIND>(t, qs, q, p.reach, &rec)) {
      weight = expected<KIND>(rec, p.cell);
      big = weight > p.leave;
      start = big ? -1 : first_fork<KIND>(t, rec);
    }
    recs[lane] = rec;
  }

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
    if (lane == 0) leaf_done = 0;
    if (mine && start >= 0)
      stack[below(alive)] = (uint32_t)lane << kOwnerShift | (uint32_t)start;
    // Hits this group may have: the lists' length, and the pool rows at hand (segments).
    int room = KIND == kBoxes && g1 - g0 > 1 ? kBoxGroupHits : kHits;
    if (KIND != kBoxes && alive) {
      const int want = min(kHits, wsum + wsum / 2 + 32);
      if (rows.end - rows.at < want) rows.refill(pool, tail, want);
      room = (int)min((long long)kHits, rows.end - rows.at);
    }
    __syncthreads();
    int sp = __popcll(alive), ncell = 0, ncand = 0, nhit = 0;
    bool over = KIND != kBoxes && alive && room == 0;  // more hits than `room`
    while (!over) {
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
          hit = cohen_sutherland<true>(a, b, bb, &cc, &dd);
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
          pool.cell[rows.at + at] = c;
          pool.xy[rows.at + at] = make_double4(cc.x, cc.y, dd.x, dd.y);
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
              pool.cell[rows.at + nhit + at] = c;
              pool.xy[rows.at + nhit + at] = make_double4(cc.x, cc.y, dd.x, dd.y);
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
      uint32_t e = lane < take ? stack[sp - take + lane] : 0;
      sp -= take;
      bool left = false, right = false;
      int child = 0, ptr = 0, size = 0;
      if (lane < take) {
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
        const bool fits = incl <= kCells - ncell && !__any(size > kLeafCells);
        uint64_t back = __ballot(size > 0 && !fits);
        const uint64_t put = __ballot(size > 0 && fits);
        if (!put) {  // the top leaf's next 64 cells; it stays on top until they are all listed
          const int top = 63 - __clzll((unsigned long long)back);
          const uint32_t done = leaf_done, cell0 = __shfl(tag | (uint32_t)ptr, top) + done;
          const uint32_t visit0 = __shfl(tag | v0, top) + done, rest = (uint32_t)__shfl(size, top) - done;
          __syncthreads();
          if ((uint32_t)lane < min(64u, rest)) cells[ncell + lane] = make_uint2(cell0 + lane, visit0 + lane);
          ncell += (int)min(64u, rest);
          if (lane == 0) leaf_done = rest > 64u ? done + 64u : 0u;
          back &= ~(1ull << top);
          if (back >> lane & 1) stack[sp + below(back)] = e;
          sp += __popcll(back);
          if (rest > 64u) {
            if (lane == top) stack[sp] = e;
            ++sp;
          }
          __syncthreads();
          continue;
        }
        if (size > 0 && fits)
          for (int j = 0; j < size; ++j)
            cells[ncell + incl - size + j] = make_uint2(tag | (uint32_t)(ptr + j), tag | (v0 + j));
        if (back >> lane & 1) stack[sp + below(back)] = e;
        sp += __popcll(back);
        // the listed cells: the prefix of the last lane that fits
        const int last = 63 - __clzll((unsigned long long)put);
        ncell += __shfl(incl, last);
      }
      __syncthreads();
    }

    bool left_over = over;  // the group's queries are left to the caller
    if (over && g1 - g0 > 1 && (KIND == kBoxes || room > 0)) {
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
    long long at = rows.at;
    if (!over && nhit > 0) {
      if constexpr (KIND == kBoxes) {
        left_over = true;
        while (left_over && rows.tried < pool.counters) {
          if (lane == 0) at = (long long)atomicAdd(rows.counter(tail), (unsigned long long)nhit);
          at = __shfl(at, 0);
          left_over = at + nhit > pool.rows;
          if (!left_over) break;
          rows.sub = rows.sub + 1 == pool.counters ? 0 : rows.sub + 1;
          ++rows.tried;
        }
        at += (long long)rows.sub * pool.rows;
        if (!left_over) {
          if (g1 - g0 > 1) {
            if (nhit <= 256) group_by_owner<4, false>(hits, nullptr, nullptr, nhit, lane, first, cnt);
            else group_by_owner<(kBoxGroupHits + 63) / 64, false>(hits, nullptr, nullptr, nhit, lane, first, cnt);
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
        if (grouped) group_by_owner<(kSegHits + 63) / 64, true>(hits, ts, byown, nhit, lane, first, cnt);
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
        rows.at += nhit;
      }
    }
    if (mine) {
      const bool leave = big || (left_over && (over ? start >= 0 : c_own > 0));
      counts[q] = leave ? 0 : c_own;
      starts[q] = leave ? -1 : at + my_first;
      if (leave) atomicAdd(reinterpret_cast<unsigned long long*>(tail), 1ull);
    }
    g0 = g1;
  }
}

// ------------------------------------------------------------------ launches
constexpr int kRowChunk = 64;  // pool rows a wavefront takes at a time, at least (segments)

inline GatherParams gather_params(const ct_tree* tree, int64_t n, const int32_t* visit, int kind) {
  GatherParams p{};
  p.visit = visit;
  p.scale(view(tree));
  // Few queries: fewer per wavefront, so that at least 4096 wavefronts share the work (256 CUs hold
  // about 4000 of them); many: 16 (8 per wavefront: 1e6 boxes 1.41 instead of 1.22
  // ms, 1e6 segments 2.74 instead of 2.67: too few entries on the stack to fill the lanes).
  p.per_wave = (int)std::min((int64_t)kMaxPerWave, std::max((int64_t)1, n / 4096));
  p.depth1 = tree->depth + 1;
  p.stack = kStack + p.depth1;
  p.group = kind == kBoxes ? kBoxGroup : kSegGroup;
  // A walk in vain costs more than leaving a query that would have fitted.
  p.leave = kind == kBoxes ? kBoxHits : kSegHits;
  return p;
}

inline Pool gather_pool(int64_t rows, int64_t n, int per_wave, int32_t* cell, double* xy, int32_t* src) {
  const int64_t waves = (n + per_wave - 1) / per_wave;
  Pool pool{cell, reinterpret_cast<double4*>(xy), src, 0, 1, kRowChunk};
  pool.counters = (int)std::min((int64_t)kPools, std::max((int64_t)1, waves / 64));
  pool.rows = rows / pool.counters;
  return pool;
}

inline int check_gather(const ct_tree* tree, int32_t kind, int64_t n) {
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

}  // namespace
}  // namespace ct

#endif  // CT_GATHER_H
