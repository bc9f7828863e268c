// ct_faces.hip -- pair-parallel FP64 polygon kernels: separating-axis test
// (separating_axis.py) and Sutherland-Hodgman clip area (sutherland_hodgman.py), one lane
// per (query face, tree face) candidate pair, both polygons in registers.
#include "ct_clip.h"
#include "ct_internal.h"
#include "ct_primitives.h"

namespace ct {
namespace {

constexpr double kFloatMax = 1.7976931348623157e308;

// separating_axis.py:17-39 extrema_projected / is_separating_axis.
template <int MA, int MB>
__device__ __forceinline__ bool separating(double nx, double ny, const P2 (&a)[MA], int la,
                                           const P2 (&b)[MB], int lb) {
  double mina = kFloatMax, maxa = -kFloatMax, minb = kFloatMax, maxb = -kFloatMax;
#pragma unroll
  for (int i = 0; i < MA; ++i) {
    if (i < la) {
      const double pr = dot(a[i].x, a[i].y, nx, ny);
      mina = pmin(mina, pr);
      maxa = pmax(maxa, pr);
    }
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if (i < lb) {
      const double pr = dot(b[i].x, b[i].y, nx, ny);
      minb = pmin(minb, pr);
      maxb = pmax(maxb, pr);
    }
  }
  return !(maxa > minb && maxb > mina);
}

// separating_axis.py:42-55 separating_axes(a, b): true when no edge normal of a separates.
template <int MA, int MB>
__device__ __forceinline__ bool no_separating_axis(const P2 (&a)[MA], int la, const P2 (&b)[MB], int lb) {
  P2 p = a[0];
#pragma unroll
  for (int i = 0; i < MA; ++i)
    if (i == la - 1) p = a[i];
#pragma unroll
  for (int i = 0; i < MA; ++i) {
    if (i < la) {
      const P2 q = a[i];
      const double nx = p.y - q.y, ny = q.x - p.x;
      p = q;
      if (!(nx == 0.0 && ny == 0.0) && separating<MA, MB>(nx, ny, a, la, b, lb)) return false;
    }
  }
  return true;
}

template <int MAXV>
__device__ __forceinline__ int load_face(const double* __restrict__ v, const int32_t* __restrict__ f, int nmax,
                                         int64_t k, P2 (&poly)[MAXV]) {
  return load_poly<MAXV>(f, nmax, k, v, poly);
}

// Whether a point c is so far inside a closed polygon (on the left of every edge that has a length)
// that no separating-axis test of it and another such polygon around c can fail.
//
// With c strictly left of every edge, the edges wind around c, and the polygon encloses a disc around c
// whose radius is c's smallest distance from the edges' lines, whatever its shape (convex or not).
// For two polygons both intervals of a projection on an axis n therefore hold the disc's, and overlap
// by 2 r |n|, where r >= kInside * scale is tested here edge by edge (|e|_1 bounds the edge's length).
// All coordinates are at most 64 * scale, so the products of a projection are rounded by less than
// 2^-52 * 128 * scale |n| and those of the test by less than 2^-50 * 128 * scale |e|: 3e-14 and 1.2e-13,
// against kInside = 1e-12.  NaN, infinities and scales whose products could underflow or overflow fail.
constexpr double kInside = 1e-12;

struct Inside {
  P2 c;
  double tol;      // kInside * scale
  double largest;  // coordinate magnitude met
  bool ok;

  __device__ __forceinline__ Inside(P2 centre, P2 vertex) : c(centre), largest(0.0) {
    const double scale = fabs(c.x) + fabs(c.y) + fabs(vertex.x - c.x) + fabs(vertex.y - c.y);
    tol = kInside * scale;
    ok = scale > 1e-100 && scale < 1e100;
  }
  __device__ __forceinline__ void edge(P2 p, P2 q) {
    const double ex = q.x - p.x, ey = q.y - p.y;
    const double d = cross(ex, ey, c.x - p.x, c.y - p.y);
    const bool point = ex == 0.0 && ey == 0.0;
    ok = ok && (point || d > tol * (fabs(ex) + fabs(ey)));
    largest = fmax(largest, fmax(fabs(p.x), fabs(p.y)));
  }
  template <int MAXV>
  __device__ __forceinline__ void polygon(const P2 (&poly)[MAXV], int len) {
    P2 p = poly[0];
#pragma unroll
    for (int i = 0; i < MAXV; ++i)
      if (i == len - 1) p = poly[i];
#pragma unroll
    for (int i = 0; i < MAXV; ++i)
      if (i < len) {
        edge(p, poly[i]);
        p = poly[i];
      }
  }
  __device__ __forceinline__ bool certain() const { return ok && largest <= 64.0 / kInside * tol; }
};

// The separating-axis test on faces in memory: no_separating_axis both ways, for the few pairs that
// need it after a clip (in registers the polygons would cost every pair a wavefront per SIMD).
struct FaceRef {
  const double* v;
  const int32_t* row;
  int len;
  __device__ __forceinline__ P2 at(int i) const { return ld_vertex(v, row[i]); }
};

__device__ __forceinline__ bool no_separating_axis(const FaceRef& a, const FaceRef& b) {
  P2 p = a.at(a.len - 1);
#pragma unroll 1
  for (int i = 0; i < a.len; ++i) {
    const P2 q = a.at(i);
    const double nx = p.y - q.y, ny = q.x - p.x;
    p = q;
    if (nx == 0.0 && ny == 0.0) continue;
    double mina = kFloatMax, maxa = -kFloatMax, minb = kFloatMax, maxb = -kFloatMax;
#pragma unroll 1
    for (int k = 0; k < a.len; ++k) {
      const P2 w = a.at(k);
      const double pr = dot(w.x, w.y, nx, ny);
      mina = pmin(mina, pr);
      maxa = pmax(maxa, pr);
    }
#pragma unroll 1
    for (int k = 0; k < b.len; ++k) {
      const P2 w = b.at(k);
      const double pr = dot(w.x, w.y, nx, ny);
      minb = pmin(minb, pr);
      maxb = pmax(maxb, pr);
    }
    if (!(maxa > minb && maxb > mina)) return false;
  }
  return true;
}

// Where a kept pair goes: keep (int64 0 / 1), or a bit of its wavefront's mask and the wavefront's count.
// Every lane of the wavefront calls this.
struct Kept {
  int64_t* keep;
  unsigned long long* masks;
  int64_t* counts;
  __device__ __forceinline__ void put(int64_t k, int64_t n, bool kept) const {
    if (masks == nullptr) {
      if (keep != nullptr && k < n) keep[k] = kept ? 1 : 0;
      return;
    }
    const uint64_t mask = __ballot(k < n && kept);
    if (lane_id() == 0 && k < n) {
      masks[k >> 6] = mask;
      counts[k >> 6] = __popcll(mask);
    }
  }
};

// Fused pair stage of locate_faces / intersect_faces (celltree.py:186-269).  Bound by the VALU.  With
// areas the clip runs first: a pair without area is dropped whatever the separating-axis test says,
// and a pair with one nearly always has the mean of the clipped polygon well inside both faces, which
// settles the test (Inside) at an eighth of its operations.  3.77e6 candidates, hexagons on triangles
// and quads: 306 -> 252 us.  Past 16 vertices together the clip runs in scratch memory and the test
// comes first: 40,000 24-gons on 20,000 triangles 926 -> 709 us.
template <int MA, int MB, bool AREA>
__global__ void __launch_bounds__(kBlock) k_face_pairs(const double* __restrict__ va,
                                                       const int32_t* __restrict__ fa, int na,
                                                       const double* __restrict__ vb,
                                                       const int32_t* __restrict__ fb, int nbm,
                                                       const int64_t* __restrict__ ii,
                                                       const int64_t* __restrict__ jj, int64_t n,
                                                       double* __restrict__ area, Kept out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool kept = false;
  if (k < n) {
    P2 a[MA], b[MB];
    int64_t i = ii[k];
    const int64_t j = jj[k];
    const int la = load_face<MA>(va, fa, na, i, a);
    const int lb = load_face<MB>(vb, fb, nbm, j, b);
    if constexpr (!AREA) {
      kept = no_separating_axis<MA, MB>(a, la, b, lb) && no_separating_axis<MB, MA>(b, lb, a, la);
    } else if constexpr (MA + MB > 16) {
      double ar = 0.0;
      if (no_separating_axis<MA, MB>(a, la, b, lb) && no_separating_axis<MB, MA>(b, lb, a, la)) {
        CT_CLIP_ROWS((clip_row_cap<MA, MB>()), row);
        ar = clip_area<MA, MB>(a, la, b, lb, row);
      }
      area[k] = ar;
      kept = ar > 0;
    } else {
      CT_CLIP_ROWS((clip_row_cap<MA, MB>()), row);
      P2 c = {0.0, 0.0};
      double ar = clip_area<MA, MB>(a, la, b, lb, row, &c);
      if (!(ar == 0.0)) {
        Inside in(c, b[0]);
        in.polygon<MB>(b, lb);
        // the subject again: kept in registers through the clip it would cost a wavefront per SIMD
        asm volatile("" : "+v"(i));
        const FaceRef fra{va, fa + i * na, la}, frb{vb, fb + j * nbm, lb};
        P2 a2[MA];
        load_face<MA>(va, fa, na, i, a2);
        in.polygon<MA>(a2, la);
        if (!in.certain() && !(no_separating_axis(fra, frb) && no_separating_axis(frb, fra))) ar = 0.0;
      }
      area[k] = ar;
      kept = ar > 0;
    }
  }
  out.put(k, n, kept);
}

// sutherland_hodgman.py:151-168 area_of_intersection (no SAT).
template <int MA, int MB>
__global__ void __launch_bounds__(kBlock) k_area(const double* __restrict__ va, const int32_t* __restrict__ fa,
                                                 int na, const double* __restrict__ vb,
                                                 const int32_t* __restrict__ fb, int nbm,
                                                 const int64_t* __restrict__ ia,
                                                 const int64_t* __restrict__ ib, int64_t n,
                                                 double* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  P2 a[MA], b[MB];
  const int la = load_face<MA>(va, fa, na, ia[k], a);
  const int lb = load_face<MB>(vb, fb, nbm, ib[k], b);
  CT_CLIP_ROWS((clip_row_cap<MA, MB>()), row);
  out[k] = clip_area<MA, MB>(a, la, b, lb, row);
}

// separating_axis.py:58-75 polygons_intersect.
template <int MA, int MB>
__global__ void __launch_bounds__(kBlock) k_sat(const double* __restrict__ va, const int32_t* __restrict__ fa,
                                                int na, const double* __restrict__ vb,
                                                const int32_t* __restrict__ fb, int nbm,
                                                const int64_t* __restrict__ ia,
                                                const int64_t* __restrict__ ib, int64_t n,
                                                uint8_t* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  P2 a[MA], b[MB];
  const int la = load_face<MA>(va, fa, na, ia[k], a);
  const int lb = load_face<MB>(vb, fb, nbm, ib[k], b);
  out[k] = (no_separating_axis<MA, MB>(a, la, b, lb) && no_separating_axis<MB, MA>(b, lb, a, la)) ? 1 : 0;
}

// sutherland_hodgman.py:171-187 box_area_of_intersection (+ celltree.py:183 area > 0):
// subject = the box as a CCW quad (geometry_utils.py:513-524), clipper = the face.
// Faces of more than 16 vertices: four wavefronts a SIMD, although the registers allow five, since their
// polygons lie in scratch and a fifth only pushes them out of the L2 (3.6e6 pairs of 24-gons 18.2 -> 17.7 ms).
template <int MB>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(MB > 16 ? 4 : 1, MB > 16 ? 4 : 8)))
k_box_pairs(const double* __restrict__ boxes,
                                                      const double* __restrict__ vb,
                                                      const int32_t* __restrict__ fb, int nbm,
                                                      const int64_t* __restrict__ ii,
                                                      const int64_t* __restrict__ jj, int64_t n,
                                                      double* __restrict__ area, Kept out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t at = k < n ? k : n - 1;  // lanes past the end repeat the last pair
  const Box bx = ld_box(boxes, ii[at]);
  const P2 a[4] = {{bx.xmin, bx.ymin}, {bx.xmax, bx.ymin}, {bx.xmax, bx.ymax}, {bx.xmin, bx.ymax}};
  P2 b[MB];
  const int lb = load_face<MB>(vb, fb, nbm, jj[at], b);
  CT_CLIP_ROWS((clip_row_cap<4, MB>()), row);
  const double ar = clip_area<4, MB>(a, 4, b, lb, row);
  if (k < n) area[k] = ar;
  out.put(k, n, ar > 0);
}

__global__ void __launch_bounds__(kBlock) k_compact(const int64_t* __restrict__ ii,
                                                    const int64_t* __restrict__ jj,
                                                    const double* __restrict__ area,
                                                    const int64_t* __restrict__ keep,
                                                    const int64_t* __restrict__ offsets, int64_t n,
                                                    int64_t* __restrict__ io, int64_t* __restrict__ jo,
                                                    double* __restrict__ ao) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n || !keep[k]) return;
  const int64_t o = offsets[k];
  io[o] = ii[k];
  jo[o] = jj[k];
  if (area && ao) ao[o] = area[k];
}

// The same from masks: a mask and the first output row per 64 pairs (3.77e6 pairs, scan and compaction:
// 80 us from int64 flags, now 41).
__global__ void __launch_bounds__(kBlock) k_compact_masks(const int64_t* __restrict__ ii, const int64_t* __restrict__ jj,
                                                          const double* __restrict__ area,
                                                          const unsigned long long* __restrict__ masks,
                                                          const int64_t* __restrict__ offsets, int64_t n,
                                                          int64_t* __restrict__ io, int64_t* __restrict__ jo,
                                                          double* __restrict__ ao) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint64_t mask = masks[k >> 6], bit = 1ull << lane_id();
  if (!(mask & bit)) return;
  const int64_t o = offsets[k >> 6] + __popcll(mask & (bit - 1));
  io[o] = ii[k];
  jo[o] = jj[k];
  if (area && ao) ao[o] = area[k];
}

inline int vclass(int nmax) { return nmax <= 4 ? 4 : nmax <= 8 ? 8 : nmax <= 16 ? 16 : 32; }

// Dispatches a pair kernel over the (subject, clipper) vertex-count classes.
template <template <int, int> class K, typename... Args>
int dispatch_pairs(int na, int nb, int64_t n, hipStream_t st, Args... args) {
  const unsigned g = grid_for(n);
  const int A = vclass(na), B = vclass(nb);
#define CT_CASE(X, Y)                                                     \
  if (A == X && B == Y) {                                                 \
    K<X, Y>::launch(g, st, args...);                                      \
    CT_LAUNCH_CHECK();                                                    \
    return CT_OK;                                                         \
  }
  CT_CASE(4, 4) CT_CASE(4, 8) CT_CASE(8, 4) CT_CASE(8, 8)
  CT_CASE(4, 16) CT_CASE(16, 4) CT_CASE(8, 16) CT_CASE(16, 8) CT_CASE(16, 16)
  CT_CASE(4, 32) CT_CASE(32, 4) CT_CASE(8, 32) CT_CASE(32, 8) CT_CASE(16, 32) CT_CASE(32, 16)
  CT_CASE(32, 32)
#undef CT_CASE
  set_error("unsupported vertex counts %d, %d", na, nb);
  return CT_ERR_ARG;
}

template <int X, int Y>
struct LFacePairs {
  template <typename... A>
  static void launch(unsigned g, hipStream_t st, A... a) {
    k_face_pairs<X, Y, false><<<g, kBlock, 0, st>>>(a...);
  }
};
template <int X, int Y>
struct LFaceAreas {
  template <typename... A>
  static void launch(unsigned g, hipStream_t st, A... a) {
    k_face_pairs<X, Y, true><<<g, kBlock, 0, st>>>(a...);
  }
};
template <int X, int Y>
struct LArea {
  template <typename... A>
  static void launch(unsigned g, hipStream_t st, A... a) {
    k_area<X, Y><<<g, kBlock, 0, st>>>(a...);
  }
};
template <int X, int Y>
struct LSat {
  template <typename... A>
  static void launch(unsigned g, hipStream_t st, A... a) {
    k_sat<X, Y><<<g, kBlock, 0, st>>>(a...);
  }
};

int launch_face_pairs(const double* va, const int32_t* fa, int na, const double* vb, const int32_t* fb, int nb,
                      const int64_t* ii, const int64_t* jj, int64_t n, int with_area, double* area, Kept out,
                      hipStream_t st) {
  if (with_area) return dispatch_pairs<LFaceAreas>(na, nb, n, st, va, fa, na, vb, fb, nb, ii, jj, n, area, out);
  return dispatch_pairs<LFacePairs>(na, nb, n, st, va, fa, na, vb, fb, nb, ii, jj, n, area, out);
}

int launch_box_pairs(const double* boxes, const double* vertices, const int32_t* faces, int nmax, const int64_t* ii,
                     const int64_t* jj, int64_t n, double* area, Kept out, hipStream_t st) {
  CT_REQUIRE(n >= 0 && nmax >= 3 && nmax <= 32, "bad sizes");
  if (n == 0) return CT_OK;
  const unsigned g = grid_for(n);
  switch (vclass(nmax)) {
    case 4: k_box_pairs<4><<<g, kBlock, 0, st>>>(boxes, vertices, faces, nmax, ii, jj, n, area, out); break;
    case 8: k_box_pairs<8><<<g, kBlock, 0, st>>>(boxes, vertices, faces, nmax, ii, jj, n, area, out); break;
    case 16: k_box_pairs<16><<<g, kBlock, 0, st>>>(boxes, vertices, faces, nmax, ii, jj, n, area, out); break;
    default: k_box_pairs<32><<<g, kBlock, 0, st>>>(boxes, vertices, faces, nmax, ii, jj, n, area, out); break;
  }
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // namespace
}  // namespace ct

using namespace ct;

extern "C" {

int ct_polygons_intersect(const double* vertices_a, const double* vertices_b, const int32_t* faces_a,
                          int32_t n_max_a, const int32_t* faces_b, int32_t n_max_b,
                          const int64_t* indices_a, const int64_t* indices_b, int64_t n, uint8_t* out,
                          void* stream) {
  CT_REQUIRE(n >= 0 && n_max_a >= 3 && n_max_b >= 3 && n_max_a <= 32 && n_max_b <= 32, "bad sizes");
  if (n == 0) return CT_OK;
  return dispatch_pairs<LSat>(n_max_a, n_max_b, n, as_stream(stream), vertices_a, faces_a, (int)n_max_a,
                              vertices_b, faces_b, (int)n_max_b, indices_a, indices_b, n, out);
}

int ct_area_of_intersection(const double* vertices_a, const double* vertices_b, const int32_t* faces_a,
                            int32_t n_max_a, const int32_t* faces_b, int32_t n_max_b,
                            const int64_t* indices_a, const int64_t* indices_b, int64_t n, double* out,
                            void* stream) {
  CT_REQUIRE(n >= 0 && n_max_a >= 3 && n_max_b >= 3 && n_max_a <= 32 && n_max_b <= 32, "bad sizes");
  if (n == 0) return CT_OK;
  return dispatch_pairs<LArea>(n_max_a, n_max_b, n, as_stream(stream), vertices_a, faces_a, (int)n_max_a,
                               vertices_b, faces_b, (int)n_max_b, indices_a, indices_b, n, out);
}

int ct_face_pairs(const double* vertices_a, const int32_t* faces_a, int32_t n_max_a,
                  const double* vertices_b, const int32_t* faces_b, int32_t n_max_b, const int64_t* ii,
                  const int64_t* jj, int64_t n, int32_t with_area, double* area, int64_t* keep,
                  void* stream) {
  CT_REQUIRE(n >= 0 && n_max_a >= 3 && n_max_b >= 3 && n_max_a <= 32 && n_max_b <= 32, "bad sizes");
  if (n == 0) return CT_OK;
  return launch_face_pairs(vertices_a, faces_a, n_max_a, vertices_b, faces_b, n_max_b, ii, jj, n, with_area, area,
                           Kept{keep, nullptr, nullptr}, as_stream(stream));
}

int ct_box_area_of_intersection(const double* bbox_coords, const double* vertices, const int32_t* faces,
                                int32_t n_max_vert, const int64_t* indices_bbox,
                                const int64_t* indices_face, int64_t n, double* out, void* stream) {
  return ct_box_pairs(bbox_coords, vertices, faces, n_max_vert, indices_bbox, indices_face, n, out,
                      nullptr, stream);
}

int ct_box_pairs(const double* bbox_coords, const double* vertices, const int32_t* faces,
                 int32_t n_max_vert, const int64_t* ii, const int64_t* jj, int64_t n, double* area,
                 int64_t* keep, void* stream) {
  return launch_box_pairs(bbox_coords, vertices, faces, n_max_vert, ii, jj, n, area, Kept{keep, nullptr, nullptr},
                          as_stream(stream));
}

int ct_face_pairs_masks(const double* vertices_a, const int32_t* faces_a, int32_t n_max_a, const double* vertices_b,
                        const int32_t* faces_b, int32_t n_max_b, const int64_t* ii, const int64_t* jj, int64_t n,
                        int32_t with_area, double* area, int64_t* masks, int64_t* counts, void* stream) {
  CT_REQUIRE(n >= 0 && n_max_a >= 3 && n_max_b >= 3 && n_max_a <= 32 && n_max_b <= 32, "bad sizes");
  if (n == 0) return CT_OK;
  CT_REQUIRE(masks && counts && (!with_area || area), "null outputs");
  return launch_face_pairs(vertices_a, faces_a, n_max_a, vertices_b, faces_b, n_max_b, ii, jj, n, with_area, area,
                           Kept{nullptr, reinterpret_cast<unsigned long long*>(masks), counts}, as_stream(stream));
}

int ct_box_pairs_masks(const double* bbox_coords, const double* vertices, const int32_t* faces, int32_t n_max_vert,
                       const int64_t* ii, const int64_t* jj, int64_t n, double* area, int64_t* masks, int64_t* counts,
                       void* stream) {
  CT_REQUIRE(n == 0 || (masks && counts && area), "null outputs");
  return launch_box_pairs(bbox_coords, vertices, faces, n_max_vert, ii, jj, n, area,
                          Kept{nullptr, reinterpret_cast<unsigned long long*>(masks), counts}, as_stream(stream));
}

int ct_compact_masks(const int64_t* ii, const int64_t* jj, const double* area, const int64_t* masks,
                     const int64_t* offsets, int64_t n, int64_t* ii_out, int64_t* jj_out, double* area_out,
                     void* stream) {
  CT_REQUIRE(n >= 0, "n must be >= 0");
  if (n == 0) return CT_OK;
  k_compact_masks<<<grid_for(n), kBlock, 0, as_stream(stream)>>>(
      ii, jj, area, reinterpret_cast<const unsigned long long*>(masks), offsets, n, ii_out, jj_out, area_out);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_compact_pairs(const int64_t* ii, const int64_t* jj, const double* area, const int64_t* keep,
                     const int64_t* offsets, int64_t n, int64_t* ii_out, int64_t* jj_out,
                     double* area_out, void* stream) {
  CT_REQUIRE(n >= 0, "n must be >= 0");
  if (n == 0) return CT_OK;
  k_compact<<<grid_for(n), kBlock, 0, as_stream(stream)>>>(ii, jj, area, keep, offsets, n, ii_out, jj_out,
                                                           area_out);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // extern "C"
