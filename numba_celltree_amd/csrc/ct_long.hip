// ct_long.hip -- box and segment queries that a wavefront walk left over (ct_gather.h): too many rows for
// its LDS lists, or no room in the pool.  A wavefront each, walked in the order of the rows, so that the
// rows need no list and there may be any number of them.
//
// The stack holds one query's nodes in the order of their leaves' positions, the first to be visited (the
// last in position: a depth-first walk that enters the right child first) on top.  A step takes the top
// 64, puts the viable children in their place, and lists the cells of the leaves at the very top, those
// with nothing before them, on a ring; the ring's cells are tested 64 at a time, as are the candidates
// that a segment's clip takes from a second ring.  A hit's row is the hits before it and those of the
// lanes below.
//
// Boxes write their cells to pool rows reserved by their expected number, or, where these do not suffice,
// by a second walk straight to the output.  Segments count, then walk again into staging rows, which
// ct_sort_staged_rows ranks by t: twice the work, but few queries, whose walks one after the other are what
// the call waits for.  Bound by the latency of a step's loads.
#include "ct_gather.h"

namespace ct {
namespace {

constexpr int kRing = 256, kCandRing = 128;
constexpr uint32_t kLeaf = 1u << 30;  // a stack entry known to be a leaf
constexpr int kLongTries = 4;         // pool counters a wavefront asks before it does without

// Walks record r from node `start` (-1: nowhere) and calls put(row, cell, piece) for every row, in the
// walk's order; returns the number of rows.  For workgroups of one wavefront.
template <int KIND, int MAXV, typename Put>
__device__ __forceinline__ int64_t ordered_walk(const TreeView& t, const QueryRec<KIND>& r, int start,
                                                const GatherParams& p, uint32_t* stack, Put put) {
  __shared__ uint32_t ring[kRing];                             // positions of listed cells
  __shared__ uint32_t cand[KIND == kFaces ? kCandRing : 1];    // segment-face: box test passed
  const int lane = lane_id();
  const P2 a = {r.d.x, r.d.y}, b = {r.d.z, r.d.w};
  int64_t rows = 0;
  int sp = start >= 0 ? 1 : 0, head = 0, nring = 0, chead = 0, ncand = 0;
  int leaf_at = 0, leaf_left = 0;  // a leaf larger than the ring: its next position, the cells left
  if (lane == 0) stack[0] = (uint32_t)start;
  __syncthreads();
  auto emit = [&](bool hit, int c, P2 cc, P2 dd) {
    const uint64_t mask = __ballot(hit);
    if (hit) put(rows + below(mask), c, cc, dd);
    rows += __popcll(mask);
  };
  while (true) {
    const bool listed_all = sp == 0 && leaf_left == 0;
    if (KIND == kFaces && (ncand >= 64 || (listed_all && nring == 0 && ncand > 0))) {
      const int m = min(64, ncand);
      bool hit = lane < m;
      int c = 0;
      P2 cc{}, dd{};
      if (hit) {
        const int k = (int)cand[(chead + lane) & (kCandRing - 1)];
        c = t.bb_indices[k];
        const Box bb = leaf_box(t, k, c);
        hit = cohen_sutherland<true>(a, b, bb, &cc, &dd);
        if (hit) {
          if (t.leaf != nullptr) hit = edge_face_clip_row<MAXV>(t, k, c, a, b, &cc, &dd);
          else hit = edge_face_clip<MAXV>(t, c, bb, a, b, &cc, &dd);
        }
      }
      chead = (chead + m) & (kCandRing - 1);
      ncand -= m;
      emit(hit, c, cc, dd);
      __syncthreads();
      continue;
    }
    if (nring >= 64 || (listed_all && nring > 0)) {
      const int m = min(64, nring);
      bool hit = lane < m;
      int k = 0, c = 0;
      P2 cc{}, dd{};
      if (hit) {
        k = (int)ring[(head + lane) & (kRing - 1)];
        hit = cell_test<KIND>(t, r, k, &c, &cc, &dd);
      }
      head = (head + m) & (kRing - 1);
      nring -= m;
      if constexpr (KIND == kFaces) {
        const uint64_t mask = __ballot(hit);
        if (hit) cand[(chead + ncand + below(mask)) & (kCandRing - 1)] = (uint32_t)k;
        ncand += __popcll(mask);
      } else {
        if constexpr (KIND == kBoxes) c = hit ? t.bb_indices[k] : 0;
        emit(hit, c, cc, dd);
      }
      __syncthreads();
      continue;
    }
    if (leaf_left > 0) {
      const int m = min(64, leaf_left);
      if (lane < m) ring[(head + nring + lane) & (kRing - 1)] = (uint32_t)(leaf_at + lane);
      nring += m;
      leaf_at += m;
      leaf_left -= m;
      __syncthreads();
      continue;
    }
    if (sp == 0) break;
    // The top of the stack: as many as their children have room for, depth + 1 places kept for a single
    // entry's way down.
    const int take = min(min(64, sp), max(1, p.stack - p.depth1 - sp));
    bool left = false, right = false, leaf = false;
    uint32_t e = 0;
    int child = 0, ptr = 0, size = 0;
    if (lane < take) {
      e = stack[sp - take + lane];
      const uint32_t x = e & ~kLeaf;
      bool here = true, by_box = false;
      NodeLd nd;
      if constexpr (KIND == kFaces) by_box = r.prune != 0;
      if ((e & kLeaf) != 0 || by_box) {
        const int4 w = ld_rec<int4>(t.nodes, x, 1);
        nd = NodeLd{0.0, 0.0, w.x, w.y, w.z, w.w};
        if constexpr (KIND == kFaces)
          if ((e & kLeaf) == 0) here = seg_near(r, ld_rec<double4>(t.nbox, x + 1));
        left = right = here && nd.child != -1;
      } else {
        const double2 lr = ld_rec<double2>(t.nodes, x);
        const int4 w = ld_rec<int4>(t.nodes, x, 1);
        nd = NodeLd{lr.x, lr.y, w.x, w.y, w.z, w.w};
        if (nd.child != -1) slab<KIND>(r, nd, &left, &right);
      }
      child = nd.child;
      if (here && child == -1 && nd.size > 0) {
        leaf = true;
        ptr = nd.ptr;
        size = nd.size;
      }
    }
    // Leaves above every entry with children: their cells come next, the topmost leaf's first.
    const uint64_t inner = __ballot(left || right);
    const bool next = leaf && (inner == 0 || lane > 63 - __clzll((unsigned long long)inner));
    int upto = next ? size : 0;  // the cells of this leaf and those above it
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_down(upto, d);
      if (lane + d < 64) upto += y;
    }
    const bool fits = next && upto <= kRing - nring;
    const uint64_t want = __ballot(next), listed = __ballot(fits);
    // the topmost, larger than the room (at least 193 cells): listed piece by piece
    const int top = 63 - __clzll((unsigned long long)(want | 1ull));
    const bool piecewise = want != 0 && listed == 0;
    if (piecewise) {
      leaf_at = __shfl(ptr, top);
      leaf_left = __shfl(size, top);
    }
    if (fits)
      for (int j = 0; j < size; ++j) ring[(head + nring + upto - size + j) & (kRing - 1)] = (uint32_t)(ptr + j);
    if (listed) nring += __shfl(upto, __ffsll((unsigned long long)listed) - 1);
    const bool stays = leaf && !fits && !(piecewise && lane == top);
    const uint64_t m1 = __ballot(left || right || stays), m2 = __ballot(left && right);
    const int to = sp - take + below(m1) + below(m2);
    __syncthreads();  // the taken entries are read
    if (stays) {
      stack[to] = e | kLeaf;
    } else if (left || right) {
      stack[to] = (uint32_t)(child + (left ? 0 : 1));
      if (left && right) stack[to + 1] = (uint32_t)(child + 1);
    }
    sp += __popcll(m1) + __popcll(m2) - take;
    __syncthreads();
  }
  return rows;
}

// The record of list entry i's query in LDS, and the node where its walk starts.
template <int KIND>
__device__ __forceinline__ int begin(const TreeView& t, const double* __restrict__ qs, int64_t q, const GatherParams& p,
                                     QueryRec<KIND>* shared) {
  QueryRec<KIND> rec;
  const int start = load_query<KIND>(t, qs, q, p.reach, &rec) ? first_fork<KIND>(t, rec) : -1;
  if (lane_id() == 0) *shared = rec;
  __syncthreads();
  return start;
}

// counts[q] of the queries in the list; boxes whose rows fit what they reserved of the pool are kept there
// (starts[q]), segments have their counts in list order too.
template <int KIND, int MAXV>
__global__ void __launch_bounds__(64, MAXV <= 8 ? 4 : 2)
k_long_count(TreeView t, const double* __restrict__ qs, const int32_t* __restrict__ left, GatherParams p, Pool pool,
             int64_t* __restrict__ counts, int64_t* __restrict__ starts, int64_t* __restrict__ left_counts,
             int64_t* tail) {
  extern __shared__ uint32_t stack[];
  __shared__ QueryRec<KIND> rec;
  const int64_t q = left[blockIdx.x];
  const int start = begin<KIND>(t, qs, q, p, &rec);
  long long at = 0, room = 0;
  if constexpr (KIND == kBoxes) {
    if (pool.rows > 0) {
      PoolRows rows;
      rows.sub = (int)(blockIdx.x % (unsigned)pool.counters);
      rows.tried = max(0, pool.counters - kLongTries);
      const int e = expected<KIND>(rec, p.cell);
      rows.refill(pool, tail, (int)min((int64_t)e + e / 4 + 64, t.n_elements));
      at = rows.at;
      room = rows.end - rows.at;
    }
  }
  const int64_t m = ordered_walk<KIND, MAXV>(t, rec, start, p, stack, [&](int64_t row, int c, P2, P2) {
    if (KIND == kBoxes && row < room) pool.cell[at + row] = c;
  });
  if (lane_id() != 0) return;
  counts[q] = m;
  if (KIND == kBoxes && room > 0 && m <= room) starts[q] = at;
  if (KIND != kBoxes) left_counts[blockIdx.x] = m;
}

// The rows of the boxes in the list that are not in the pool.
__global__ void __launch_bounds__(64, 4)
k_long_boxes(TreeView t, const double* __restrict__ boxes, const int32_t* __restrict__ left, GatherParams p,
             const int64_t* __restrict__ offsets, const int64_t* __restrict__ starts, int64_t* __restrict__ ii,
             int64_t* __restrict__ jj) {
  extern __shared__ uint32_t stack[];
  __shared__ QueryRec<kBoxes> rec;
  const int64_t q = left[blockIdx.x];
  if (starts[q] >= 0) return;
  const int start = begin<kBoxes>(t, boxes, q, p, &rec);
  const int64_t o = offsets[q];
  ordered_walk<kBoxes, 4>(t, rec, start, p, stack, [&](int64_t row, int c, P2, P2) {
    ii[o + row] = q;
    jj[o + row] = c;
  });
}

// The rows of the segments in the list into staging, in list order; starts[q]: the first.
template <int KIND, int MAXV>
__global__ void __launch_bounds__(64, MAXV <= 8 ? 4 : 2)
k_long_edges(TreeView t, const double* __restrict__ segs, const int32_t* __restrict__ left, GatherParams p,
             const int64_t* __restrict__ left_offsets, int64_t* __restrict__ starts, StagedRows rows) {
  extern __shared__ uint32_t stack[];
  __shared__ QueryRec<KIND> rec;
  const int64_t q = left[blockIdx.x];
  const int start = begin<KIND>(t, segs, q, p, &rec);
  const int64_t o = left_offsets[blockIdx.x];
  if (lane_id() == 0) starts[q] = o;
  ordered_walk<KIND, MAXV>(t, rec, start, p, stack, [&](int64_t row, int c, P2 cc, P2 dd) {
    rows.query[o + row] = (int32_t)q;
    rows.cell[o + row] = c;
    rows.xy[o + row] = make_double4(cc.x, cc.y, dd.x, dd.y);
    rows.t[o + row] = row_t(rec.d, make_double2(cc.x, cc.y));
  });
}

int check_long(const ct_tree* tree, int32_t kind, int64_t n, int64_t n_left) {
  const int rc = check_gather(tree, kind, n);
  if (rc) return rc;
  CT_REQUIRE(n_left >= 0 && n_left <= n && n_left <= CT_LONG_MAX, "at most %d queries left", (int)CT_LONG_MAX);
  return CT_OK;
}

}  // namespace
}  // namespace ct

using namespace ct;

extern "C" {

int ct_long_count(const ct_tree* tree, int32_t kind, const double* queries, int64_t n, const int32_t* left,
                  int64_t n_left, int64_t pool_rows, int32_t* pool_cell, int64_t* counts, int64_t* starts,
                  int64_t* left_counts, int64_t* tail, void* stream) {
  const int rc = check_long(tree, kind, n, n_left);
  if (rc) return rc;
  CT_REQUIRE(n_left == 0 || (queries && left && counts && starts && tail && (kind == kBoxes || left_counts)),
             "null pointer");
  CT_REQUIRE(pool_rows >= 0 && pool_rows < ((int64_t)1 << 31) && (pool_rows == 0 || pool_cell), "bad pool");
  if (n_left == 0) return CT_OK;
  const TreeView t = view(tree);
  const GatherParams p = gather_params(tree, n, nullptr, kind);
  const Pool pool = gather_pool(kind == kBoxes ? pool_rows : 0, n, p.per_wave, pool_cell, nullptr, nullptr);
  hipStream_t st = as_stream(stream);
  const unsigned g = (unsigned)n_left;
  const size_t lds = p.stack * sizeof(uint32_t);
  const int nm = tree->n_max_vert;
#define CT_LONG(KIND, MAXV) \
  k_long_count<KIND, MAXV><<<g, 64, lds, st>>>(t, queries, left, p, pool, counts, starts, left_counts, tail)
  if (kind == kBoxes) CT_LONG(kBoxes, 4);
  else if (kind == kEdges) CT_LONG(kEdges, 4);
  else if (nm <= 4) CT_LONG(kFaces, 4);
  else if (nm <= 8) CT_LONG(kFaces, 8);
  else if (nm <= 16) CT_LONG(kFaces, 16);
  else CT_LONG(kFaces, 32);
#undef CT_LONG
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_long_boxes(const ct_tree* tree, const double* boxes, int64_t n, const int32_t* left, int64_t n_left,
                  const int64_t* offsets, const int64_t* starts, int64_t* ii, int64_t* jj, void* stream) {
  const int rc = check_long(tree, kBoxes, n, n_left);
  if (rc) return rc;
  CT_REQUIRE(n_left == 0 || (boxes && left && offsets && starts && ii && jj), "null pointer");
  if (n_left == 0) return CT_OK;
  const GatherParams p = gather_params(tree, n, nullptr, kBoxes);
  k_long_boxes<<<(unsigned)n_left, 64, p.stack * sizeof(uint32_t), as_stream(stream)>>>(view(tree), boxes, left, p,
                                                                                      offsets, starts, ii, jj);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_long_edges(const ct_tree* tree, int32_t kind, const double* segments, int64_t n, const int32_t* left,
                  int64_t n_left, const int64_t* left_offsets, int64_t* starts, int32_t* rows_query,
                  int32_t* rows_cell, double* rows_xy, double* rows_t, void* stream) {
  const int rc = check_long(tree, kind, n, n_left);
  if (rc) return rc;
  CT_REQUIRE(kind != kBoxes, "kind must be 2 (segment-face) or 3 (segment-edge)");
  CT_REQUIRE(n_left == 0 || (segments && left && left_offsets && starts && rows_query && rows_cell && rows_xy && rows_t),
             "null pointer");
  if (n_left == 0) return CT_OK;
  const TreeView t = view(tree);
  const GatherParams p = gather_params(tree, n, nullptr, kind);
  const StagedRows rows{rows_query, rows_cell, reinterpret_cast<double4*>(rows_xy), rows_t, {}};
  hipStream_t st = as_stream(stream);
  const unsigned g = (unsigned)n_left;
  const size_t lds = p.stack * sizeof(uint32_t);
  const int nm = tree->n_max_vert;
#define CT_LONG(KIND, MAXV) k_long_edges<KIND, MAXV><<<g, 64, lds, st>>>(t, segments, left, p, left_offsets, starts, rows)
  if (kind == kEdges) CT_LONG(kEdges, 4);
  else if (nm <= 4) CT_LONG(kFaces, 4);
  else if (nm <= 8) CT_LONG(kFaces, 8);
  else if (nm <= 16) CT_LONG(kFaces, 16);
  else CT_LONG(kFaces, 32);
#undef CT_LONG
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // extern "C"
