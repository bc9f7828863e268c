// ct_geometry.hip -- per-element geometry kernels that prepare a tree: counter-clockwise
// reordering, face / edge bounding boxes, and the bbox statistics (tree bbox, diagonals,
// default tolerance).  One lane per element; all FP64.
#include "ct_internal.h"
#include "ct_primitives.h"

namespace ct {

// geometry_utils.py:541-561 counter_clockwise.  a = v[len-2], b = v[len-1] are fixed
// once; the loop walks the *current* row, so after a flip it reads the reversed row and
// may flip again.  The row is kept in registers and each flip toggles a parity bit:
// current[i] = parity ? orig[len-1-i] : orig[i].
template <int MAXV>
__global__ void __launch_bounds__(kBlock) k_counter_clockwise(const double* __restrict__ vertices,
                                                              int32_t* __restrict__ faces,
                                                              int64_t n_faces, int nmax) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= n_faces) return;
  int32_t* row = faces + f * nmax;
  int32_t idx[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) idx[i] = (i < nmax) ? row[i] : kFill;
  int len = nmax;
#pragma unroll
  for (int i = MAXV - 1; i >= 3; --i)
    if (i < nmax && idx[i] == kFill) len = i;

  auto vtx = [&](int i) { return ld_vertex(vertices, idx[i]); };
  P2 a = {0, 0}, b = {0, 0};
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    if (i == len - 2) a = vtx(i);
    if (i == len - 1) b = vtx(i);
  }
  bool parity = false;
  for (int i = 0; i < len; ++i) {
    const int src = parity ? (len - 1 - i) : i;
    int vi = idx[0];
#pragma unroll
    for (int j = 0; j < MAXV; ++j)
      if (j == src) vi = idx[j];
    const P2 c = ld_vertex(vertices, vi);
    const double product = cross(b.x - a.x, b.y - a.y, c.x - a.x, c.y - a.y);
    if (product == 0) {
      a = b;
      b = c;
    } else if (product < 0) {
      parity = !parity;
    } else {
      break;
    }
  }
  if (parity) {
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      if (i < len) {
        int v = idx[0];
#pragma unroll
        for (int j = 0; j < MAXV; ++j)
          if (j == len - 1 - i) v = idx[j];
        row[i] = v;
      }
    }
  }
}

// geometry_utils.py:421-456 bounding_box / build_face_bboxes: the first vertex seeds the
// box and the scan stops at the first fill value.
__global__ void __launch_bounds__(kBlock) k_face_bboxes(const int32_t* __restrict__ faces,
                                                        int64_t n_faces, int nmax,
                                                        const double* __restrict__ vertices,
                                                        double* __restrict__ out) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= n_faces) return;
  const int32_t* row = faces + f * nmax;
  const P2 v0 = ld_vertex(vertices, row[0]);
  double xmin = v0.x, xmax = v0.x, ymin = v0.y, ymax = v0.y;
  for (int i = 1; i < nmax; ++i) {
    const int32_t k = row[i];
    if (k == kFill) break;
    const P2 v = ld_vertex(vertices, k);
    xmin = pmin(xmin, v.x);
    xmax = pmax(xmax, v.x);
    ymin = pmin(ymin, v.y);
    ymax = pmax(ymax, v.y);
  }
  reinterpret_cast<double4*>(out)[f] = make_double4(xmin, xmax, ymin, ymax);
}

// geometry_utils.py:459-487 edge_bounding_box / build_edge_bboxes (padded by tol).
__global__ void __launch_bounds__(kBlock) k_edge_bboxes(const int32_t* __restrict__ edges,
                                                        int64_t n, const double* __restrict__ vertices,
                                                        double tol, double* __restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const P2 p = ld_vertex(vertices, edges[2 * e]);
  const P2 q = ld_vertex(vertices, edges[2 * e + 1]);
  reinterpret_cast<double4*>(out)[e] =
      make_double4(pmin(p.x - tol, q.x - tol), pmax(p.x + tol, q.x + tol),
                   pmin(p.y - tol, q.y - tol), pmax(p.y + tol, q.y + tol));
}

// Reductions over all cells / vertices use a bounded grid (grid-stride loops) and one atomic
// per key per workgroup: one atomic per key per wavefront on the same five addresses
// serialises at the memory side (~0.9 ms for 1M cells).
constexpr unsigned kReduceGrid = 1024;

inline unsigned reduce_grid(int64_t n) {
  const unsigned g = grid_for(n);
  return g < kReduceGrid ? g : kReduceGrid;
}

// Max of K keys over the workgroup (wavefront shuffles, then LDS across the waves), then one
// atomicMax per key.
template <int K>
__device__ __forceinline__ void block_max_atomic(unsigned long long (&k)[K], unsigned long long* __restrict__ keys) {
  __shared__ unsigned long long part[kBlock / 64][K];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const unsigned long long t = __shfl_xor(k[j], d, 64);
      k[j] = t > k[j] ? t : k[j];
    }
  }
  const int w = threadIdx.x / 64;
  if (lane_id() == 0) {
#pragma unroll
    for (int j = 0; j < K; ++j) part[w][j] = k[j];
  }
  __syncthreads();
  if (threadIdx.x < K) {
    unsigned long long m = 0;
    for (int v = 0; v < (int)(blockDim.x / 64); ++v) m = part[v][threadIdx.x] > m ? part[v][threadIdx.x] : m;
    atomicMax(keys + threadIdx.x, m);
  }
}

// celltree_base.py:20-48: per-cell dx, dy, dxy = sqrt(dx**2 + dy**2) and the tree bbox /
// maximum diagonal as order-preserving keys (keys[0..4] = min x, max x, min y, max y,
// max dxy; min slots hold negated-order keys so one atomicMax serves all five).
__global__ void __launch_bounds__(kBlock) k_bbox_stats(const double* __restrict__ bb, int64_t n,
                                                       double* __restrict__ dist,
                                                       unsigned long long* __restrict__ keys) {
  unsigned long long k[5] = {0, 0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const Box b = ld_box(bb, i);
    const double dx = b.xmax - b.xmin;
    const double dy = b.ymax - b.ymin;
    const double dxy = sqrt(dx * dx + dy * dy);
    if (dist) {
      dist[3 * i] = dx;
      dist[3 * i + 1] = dy;
      dist[3 * i + 2] = dxy;
    }
    const unsigned long long c[5] = {~dkey(b.xmin), dkey(b.xmax), ~dkey(b.ymin), dkey(b.ymax), dkey(dxy)};
#pragma unroll
    for (int j = 0; j < 5; ++j) k[j] = c[j] > k[j] ? c[j] : k[j];
  }
  block_max_atomic<5>(k, keys);
}

// A caller's face rows made ready in one pass: converted to int32 with the fill value as -1,
// checked, reordered counter-clockwise, with their boxes, box distances and the reductions of
// k_bbox_stats.  Bound by memory latency (index row, then vertices); as separate passes (a cast,
// three reductions with their host round trip, a cast, k_counter_clockwise, k_face_bboxes,
// k_bbox_stats) the same rows were read eight times: the constructor went from 1.42 to 1.26 ms at
// 999,941 cells (this pass 49 us) and from 0.43 to 0.35 ms at 20,000, intersect_faces with 250,000
// target faces from 0.84 to 0.76 ms.
//
// Every index is checked here and reported through `checks` (max, min, min of the first three
// columns), which the host reads with its next synchronization; an index that fails a check is
// replaced by 0, so that no kernel of the call reads outside the vertices before the host raises.
// checks: 8 keys reduced from 0 by maximum: signed indices as order-preserving unsigned keys
// (minima complemented), then the 5 keys of k_bbox_stats.
__device__ __forceinline__ unsigned long long ikey(int64_t v) {
  return (unsigned long long)v ^ 0x8000000000000000ull;
}

template <int MAXV, bool EXACT, typename IN>
__global__ void __launch_bounds__(kBlock) k_prepare_faces(const IN* __restrict__ in, int64_t n, int nmax_, int64_t fill,
                                                          int64_t n_vertices, const double* __restrict__ vertices,
                                                          int32_t* __restrict__ faces, double* __restrict__ bb,
                                                          double* __restrict__ dist,
                                                          unsigned long long* __restrict__ checks) {
  const int nmax = EXACT ? MAXV : nmax_;
  unsigned long long k[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < n; f += stride) {
    int32_t idx[MAXV];
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      if (i >= nmax) {
        idx[i] = kFill;
        continue;
      }
      int64_t v = (int64_t)in[f * nmax + i];
      if (v == fill) v = kFill;
      const unsigned long long u = ikey(v);
      k[0] = u > k[0] ? u : k[0];
      k[1] = ~u > k[1] ? ~u : k[1];
      if (i < 3) k[2] = ~u > k[2] ? ~u : k[2];
      if (v >= n_vertices || v < (i < 3 ? 0 : kFill)) v = 0;
      idx[i] = (int32_t)v;
    }
    int len = nmax;
#pragma unroll
    for (int i = MAXV - 1; i >= 3; --i)
      if (i < nmax && idx[i] == kFill) len = i;
    P2 p[MAXV];
#pragma unroll
    for (int i = 0; i < MAXV; ++i) p[i] = i < len ? ld_vertex(vertices, idx[i]) : P2{0.0, 0.0};
    // k_counter_clockwise on registers
    P2 a = p[0], b = p[0];
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      if (i == len - 2) a = p[i];
      if (i == len - 1) b = p[i];
    }
    bool parity = false;
    for (int i = 0; i < len; ++i) {
      const int src = parity ? (len - 1 - i) : i;
      P2 c = p[0];
#pragma unroll
      for (int j = 1; j < MAXV; ++j)
        if (j == src) c = p[j];
      const double product = cross(b.x - a.x, b.y - a.y, c.x - a.x, c.y - a.y);
      if (product == 0) {
        a = b;
        b = c;
      } else if (product < 0) {
        parity = !parity;
      } else {
        break;
      }
    }
    if (parity) {
      int32_t q[MAXV];
      P2 r[MAXV];
#pragma unroll
      for (int i = 0; i < MAXV; ++i) {
        q[i] = idx[i];
        r[i] = p[i];
#pragma unroll
        for (int j = 0; j < MAXV; ++j)
          if (i < len && j == len - 1 - i) {
            q[i] = idx[j];
            r[i] = p[j];
          }
      }
#pragma unroll
      for (int i = 0; i < MAXV; ++i) {
        idx[i] = q[i];
        p[i] = r[i];
      }
    }
    if constexpr (EXACT && MAXV == 4) {
      reinterpret_cast<int4*>(faces)[f] = make_int4(idx[0], idx[1], idx[2], idx[3]);
    } else {
#pragma unroll
      for (int i = 0; i < MAXV; ++i)
        if (i < nmax) faces[f * nmax + i] = idx[i];
    }
    // k_face_bboxes on registers (the scan stops at the first fill value, which is at len)
    double xmin = p[0].x, xmax = p[0].x, ymin = p[0].y, ymax = p[0].y;
#pragma unroll
    for (int i = 1; i < MAXV; ++i) {
      if (i >= len) break;
      xmin = pmin(xmin, p[i].x);
      xmax = pmax(xmax, p[i].x);
      ymin = pmin(ymin, p[i].y);
      ymax = pmax(ymax, p[i].y);
    }
    reinterpret_cast<double4*>(bb)[f] = make_double4(xmin, xmax, ymin, ymax);
    const double dx = xmax - xmin, dy = ymax - ymin;
    const double dxy = sqrt(dx * dx + dy * dy);
    if (dist) {
      dist[3 * f] = dx;
      dist[3 * f + 1] = dy;
      dist[3 * f + 2] = dxy;
    }
    const unsigned long long c[5] = {~dkey(xmin), dkey(xmax), ~dkey(ymin), dkey(ymax), dkey(dxy)};
#pragma unroll
    for (int j = 0; j < 5; ++j) k[3 + j] = c[j] > k[3 + j] ? c[j] : k[3 + j];
  }
  block_max_atomic<8>(k, checks);
}

template <typename IN>
int launch_prepare(const IN* in, int64_t n, int nmax, int64_t fill_value, int64_t n_vertices, const double* vertices,
                   int32_t* faces, double* bb, double* dist, unsigned long long* checks, hipStream_t st) {
  const unsigned g = reduce_grid(n);
  if (nmax == 3)
    k_prepare_faces<3, true><<<g, kBlock, 0, st>>>(in, n, nmax, fill_value, n_vertices, vertices, faces, bb, dist, checks);
  else if (nmax == 4)
    k_prepare_faces<4, true><<<g, kBlock, 0, st>>>(in, n, nmax, fill_value, n_vertices, vertices, faces, bb, dist, checks);
  else
    k_prepare_faces<8, false><<<g, kBlock, 0, st>>>(in, n, nmax, fill_value, n_vertices, vertices, faces, bb, dist, checks);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

// edge_celltree.py:60-64: extent of the vertices.
__global__ void __launch_bounds__(kBlock) k_vertex_extent(const double* __restrict__ v, int64_t n,
                                                          unsigned long long* __restrict__ keys) {
  unsigned long long k[4] = {0, 0, 0, 0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const P2 p = ld_vertex(v, (int)i);
    const unsigned long long c[4] = {~dkey(p.x), dkey(p.x), ~dkey(p.y), dkey(p.y)};
#pragma unroll
    for (int j = 0; j < 4; ++j) k[j] = c[j] > k[j] ? c[j] : k[j];
  }
  block_max_atomic<4>(k, keys);
}

__global__ void k_extent_finish(const unsigned long long* __restrict__ keys, double* __restrict__ out) {
  const int i = threadIdx.x;
  if (i < 4) out[i] = dval((i % 2 == 0) ? ~keys[i] : keys[i]);
}

__global__ void k_stats_finish(const unsigned long long* __restrict__ keys, double* __restrict__ out) {
  const int i = threadIdx.x;
  if (i < 5) out[i] = dval((i == 0 || i == 2) ? ~keys[i] : keys[i]);
}

int bbox_stat_keys(const double* bb, int64_t n, double* distances, unsigned long long* keys, hipStream_t st) {
  int rc = fill<unsigned long long>(keys, 5, 0ull, st);
  if (rc) return rc;
  k_bbox_stats<<<reduce_grid(n), kBlock, 0, st>>>(bb, n, distances, keys);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // namespace ct

using namespace ct;

extern "C" {

int ct_counter_clockwise(const double* vertices, int32_t* faces, int64_t n_faces,
                         int32_t n_max_vert, void* stream) {
  CT_REQUIRE(n_faces >= 0, "n_faces must be >= 0");
  CT_REQUIRE(n_max_vert >= 3 && n_max_vert <= CT_MAX_N_VERTEX, "n_max_vert must be in [3, 32]");
  if (n_faces == 0) return CT_OK;
  hipStream_t st = as_stream(stream);
  const unsigned g = grid_for(n_faces);
  if (n_max_vert <= 4) k_counter_clockwise<4><<<g, kBlock, 0, st>>>(vertices, faces, n_faces, n_max_vert);
  else if (n_max_vert <= 8) k_counter_clockwise<8><<<g, kBlock, 0, st>>>(vertices, faces, n_faces, n_max_vert);
  else if (n_max_vert <= 16) k_counter_clockwise<16><<<g, kBlock, 0, st>>>(vertices, faces, n_faces, n_max_vert);
  else k_counter_clockwise<32><<<g, kBlock, 0, st>>>(vertices, faces, n_faces, n_max_vert);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_build_face_bboxes(const int32_t* faces, int64_t n_faces, int32_t n_max_vert,
                         const double* vertices, double* out, void* stream) {
  CT_REQUIRE(n_faces >= 0 && n_max_vert >= 1, "bad sizes");
  if (n_faces == 0) return CT_OK;
  k_face_bboxes<<<grid_for(n_faces), kBlock, 0, as_stream(stream)>>>(faces, n_faces, n_max_vert,
                                                                      vertices, out);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_build_edge_bboxes(const int32_t* edges, int64_t n_edges, const double* vertices, double tol,
                         double* out, void* stream) {
  CT_REQUIRE(n_edges >= 0, "bad sizes");
  if (n_edges == 0) return CT_OK;
  k_edge_bboxes<<<grid_for(n_edges), kBlock, 0, as_stream(stream)>>>(edges, n_edges, vertices, tol,
                                                                      out);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_prepare_faces(const void* faces_in, int32_t index_bytes, int64_t n_faces, int32_t n_max_vert,
                     int64_t fill_value, int64_t n_vertices, const double* vertices, int32_t* faces_out,
                     double* bb_out, double* distances, uint64_t* checks, void* stream) {
  CT_REQUIRE(n_faces >= 1 && n_vertices >= 1, "need at least one face and one vertex");
  CT_REQUIRE(n_max_vert >= 3 && n_max_vert <= 8, "n_max_vert must be in [3, 8]");
  CT_REQUIRE(index_bytes == 4 || index_bytes == 8, "int32 or int64 indices");
  CT_REQUIRE(faces_in && vertices && faces_out && bb_out && checks, "null pointer");
  hipStream_t st = as_stream(stream);
  unsigned long long* keys = reinterpret_cast<unsigned long long*>(checks);
  int rc = fill<unsigned long long>(keys, 8, 0ull, st);
  if (rc) return rc;
  // an index that int32 cannot hold fails the check whatever the vertex count
  const int64_t nv = n_vertices < ((int64_t)1 << 31) ? n_vertices : ((int64_t)1 << 31);
  if (index_bytes == 4)
    return launch_prepare(static_cast<const int32_t*>(faces_in), n_faces, n_max_vert, fill_value, nv, vertices,
                          faces_out, bb_out, distances, keys, st);
  return launch_prepare(static_cast<const int64_t*>(faces_in), n_faces, n_max_vert, fill_value, nv, vertices,
                        faces_out, bb_out, distances, keys, st);
}

int ct_bbox_stats(const double* bb_coords, int64_t n, double* distances, double* out5,
                  void* stream) {
  CT_REQUIRE(n > 0, "need at least one bounding box");
  hipStream_t st = as_stream(stream);
  // out5 doubles as the key scratch: 5 keys are reduced in place, then decoded.
  unsigned long long* keys = reinterpret_cast<unsigned long long*>(out5);
  int rc = bbox_stat_keys(bb_coords, n, distances, keys, st);
  if (rc) return rc;
  k_stats_finish<<<1, 64, 0, st>>>(keys, out5);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_vertex_extent(const double* vertices, int64_t n, double* out4, void* stream) {
  CT_REQUIRE(n > 0, "need at least one vertex");
  hipStream_t st = as_stream(stream);
  unsigned long long* keys = reinterpret_cast<unsigned long long*>(out4);
  int rc = fill<unsigned long long>(keys, 4, 0ull, st);
  if (rc) return rc;
  k_vertex_extent<<<reduce_grid(n), kBlock, 0, st>>>(vertices, n, keys);
  CT_LAUNCH_CHECK();
  k_extent_finish<<<1, 64, 0, st>>>(keys, out4);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // extern "C"
