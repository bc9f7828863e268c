// ct_build.hip -- GPU build of the Garth-Joy bucket-split cell tree.
//
// The reference (creation.py:233-381) builds serially with a DFS stack.  Each node's work
// depends only on its own cell range, so the nodes can be split in any order.  Two stages:
//
//   large nodes (more cells than one workgroup holds), level by level, three kernels a level:
//     k_tile_count    per tile (<= kTile cells of ONE node): each cell's bucket, and the tile's
//                     bucket counts and bucket bounds in both dimensions
//     k_node_decide   per node: tile counts -> stable offsets, bucket bounds -> split (or
//                     retry, or leaf); the children's extents are unions of bucket bounds, so no
//                     pass over the cells computes them
//     k_tile_scatter  per tile: the stably partitioned permutation
//   small nodes (<= T cells): k_small, one workgroup per node, builds the whole subtree in LDS
//   k_top             DFS ranks and tight boxes of the large nodes, in one workgroup
//   k_emit            nodes (and tight boxes) to their reference indices
//
// What bounds it: the work per level is small (a permutation index, a 32-byte box and a byte per
// cell), so a build is made of latencies: kernel boundaries, barriers, host round trips.  Half of
// the levels lie below 1024 cells, where a workgroup's barriers replace kernel boundaries.  The
// host launches as many large-node levels as a balanced tree has, plus two, without reading
// anything back (an idle level costs three empty launches), and synchronizes once.  With a
// sequence of 11 kernels and a host synchronization for each of the 22 levels, and the node boxes
// in one launch a level, the constructor took 5.78 ms for 999,941 cells and 1.67 ms for 20,000;
// now 1.14 and 0.33 ms.
//
// The stable partition is the order sort_bbox_indices (:54-151) produces with its repeated
// stable_partition.  Per node as in the reference: special case (:312-320), empty-bucket merge
// (:322-341), retry-other-dimension / degenerate leaf (:343-358), split_plane (:174-213),
// children (:365-379).
//
// Nodes are first numbered in creation order.  The reference's DFS numbering puts the children
// of the k-th internal node in DFS preorder (left first) at 1 + 2k (creation.py:373-379): a
// bottom-up count of internal nodes per subtree and a top-down prefix give every node its
// index, and a subtree whose root has rank r occupies the indices 2r + (its own numbering).
//
// Order-sensitive details kept from the reference: FP64 bucket bounds i*bl + Rmin and
// (i+1)*bl + Rmin (no FMA), first strict minimum of the split cost, a node that retries
// keeps its flipped dim even when it ends as a leaf.
#include <algorithm>

#include "ct_internal.h"
#include "ct_primitives.h"

namespace ct {
namespace {

using Key = unsigned long long;

// Cells per tile of the large-node kernels: 4 per lane keep the tile count (and the prefix that
// k_node_decide forms over a node's tiles) low; 999,941 cells are 977 workgroups.
constexpr int kTileItems = 4;
constexpr int kTile = kBlock * kTileItems;
constexpr int kDecideBlock = 512;
constexpr int kMaxBuckets = 64;

// Cells a workgroup's subtree stage takes, by bucket count: its LDS holds per-bucket bounds of
// up to T / 2 nodes.
int small_cells(int nb) { return nb <= 8 ? 1024 : nb <= 16 ? 512 : nb <= 32 ? 256 : 128; }

struct Slots {  // large nodes of one level, structure of arrays
  int32_t* id;     // creation-order node id
  int32_t* ptr;
  int32_t* size;
  int32_t* dim;
  int32_t* att;    // 0 first attempt, 1 after a dimension flip
  int32_t* depth;
  int32_t* tile0;  // first tile; tiles of a node are consecutive
  Key* range;      // 4 per node: min x, max x, min y, max y of its cells' boxes
  int32_t* map;    // tile -> slot
};

struct Smalls {  // roots of the subtrees k_small builds
  int32_t* id;
  int32_t* ptr;
  int32_t* size;
  int32_t* dim;
  int32_t* depth;
};

// Read back by the host in one transfer.
struct Header {
  // counters that k_node_decide raises together: one 64-bit atomic instead of several on the few
  // addresses that all nodes of a level meet at (11 ns each)
  int32_t next_id;    // nodes created by the large-node stage (and the root)
  int32_t n_small;
  struct {
    int32_t active;   // large nodes
    int32_t tiles;    // and their tiles
  } level[2];         // per level parity
  int32_t err;        // 1: a centroid in no bucket, 2: no finite split cost
  int32_t depth;
  int32_t n_nodes;    // of the whole tree (k_top)
  int32_t pad[3];
  Key checks[3];      // of ct_prepare_faces, passed through
  Key stats[5];       // as bbox_stat_keys leaves them: ~min x, max x, ~min y, max y, max diagonal
};

struct Work {
  Header* head;
  int32_t* perm[2];
  uint8_t* bid;
  int32_t* tilecnt;   // per tile and bucket: cells
  int32_t* tilepre;   // per tile and bucket: cells of the node's earlier tiles
  Key* tilebk;        // per tile, bucket: 4 bounds
  int32_t* boff;      // per slot and bucket: first position
  Slots act[2];
  Smalls small;
  int32_t* group_end;  // creation-order ids at the start of every large-node level
  ct_node* cnodes;     // large-node stage, creation order; child -2: a subtree k_small built
  int32_t* icount;
  int32_t* drank;
  int32_t* newidx;
  double4* tbox;
  ct_node* lnodes;     // subtrees: node x of the subtree at positions [p, ...) is entry 2p + x
  int32_t* lmeta;      // its own DFS index | its internal rank << 16
  double4* lbox;
};

struct Layout {
  size_t bytes = 0;
  template <typename T>
  size_t take(size_t count) {
    size_t off = (bytes + 255) & ~size_t(255);
    bytes = off + count * sizeof(T);
    return off;
  }
};

// Large nodes of a level hold more than small_cells(nb) cells each.
int64_t max_active(int64_t n, int nb) { return n / (small_cells(nb) + 1) + 2; }
int64_t max_tiles(int64_t n, int nb) { return n / kTile + max_active(n, nb) + 2; }

// Carves the workspace; with base == nullptr it only measures.
Work carve(char* base, int64_t n, int nb, size_t* total) {
  Layout L;
  Work w{};
  const int64_t amax = max_active(n, nb), tmax = max_tiles(n, nb), smax = n / 2 + 2;
  const int64_t mmax = ct_max_nodes(n) + 2;
  auto P = [&](size_t off) { return base ? base + off : nullptr; };
#define CT_TAKE(field, T, count) field = reinterpret_cast<T*>(P(L.take<T>(count)))
  CT_TAKE(w.head, Header, 1);
  CT_TAKE(w.perm[0], int32_t, n);
  CT_TAKE(w.perm[1], int32_t, n);
  CT_TAKE(w.bid, uint8_t, n);
  CT_TAKE(w.tilecnt, int32_t, tmax * nb);
  CT_TAKE(w.tilepre, int32_t, tmax * nb);
  CT_TAKE(w.tilebk, Key, tmax * nb * 4);
  CT_TAKE(w.boff, int32_t, amax * nb);
  for (int k = 0; k < 2; ++k) {
    CT_TAKE(w.act[k].id, int32_t, amax);
    CT_TAKE(w.act[k].ptr, int32_t, amax);
    CT_TAKE(w.act[k].size, int32_t, amax);
    CT_TAKE(w.act[k].dim, int32_t, amax);
    CT_TAKE(w.act[k].att, int32_t, amax);
    CT_TAKE(w.act[k].depth, int32_t, amax);
    CT_TAKE(w.act[k].tile0, int32_t, amax);
    CT_TAKE(w.act[k].range, Key, amax * 4);
    CT_TAKE(w.act[k].map, int32_t, tmax);
  }
  CT_TAKE(w.small.id, int32_t, smax);
  CT_TAKE(w.small.ptr, int32_t, smax);
  CT_TAKE(w.small.size, int32_t, smax);
  CT_TAKE(w.small.dim, int32_t, smax);
  CT_TAKE(w.small.depth, int32_t, smax);
  CT_TAKE(w.group_end, int32_t, 2 * n + 8);
  CT_TAKE(w.cnodes, ct_node, mmax);
  CT_TAKE(w.icount, int32_t, mmax);
  CT_TAKE(w.drank, int32_t, mmax);
  CT_TAKE(w.newidx, int32_t, mmax);
  CT_TAKE(w.tbox, double4, mmax);
  CT_TAKE(w.lnodes, ct_node, 2 * n + 2);
  CT_TAKE(w.lmeta, int32_t, 2 * n + 2);
  CT_TAKE(w.lbox, double4, 2 * n + 2);
#undef CT_TAKE
  *total = L.bytes + 256;
  return w;
}

__device__ __forceinline__ double4 ld_box4(const double* __restrict__ bb, int c) {
  return reinterpret_cast<const double4*>(bb)[c];
}

// creation.py:44-51 + the first-match bucket of sort_bbox_indices (:115-151).  Buckets
// [i*bl + Rmin, (i+1)*bl + Rmin) share their bounding expressions, so the first matching
// bucket is the only one.  No match (-1): the reference indexes past its bucket list (error).
__device__ __forceinline__ int bucket_of(double lo, double hi, double range_Rmin, double bl, int nb) {
  const double centroid = lo + 0.5 * (hi - lo);
  for (int k = 0; k < nb; ++k) {
    const double bmax = (double)(k + 1) * bl + range_Rmin;  // creation.py:286
    const double bmin = (double)k * bl + range_Rmin;        // creation.py:287
    if ((centroid >= bmin) && (centroid < bmax)) return k;
  }
  return -1;
}

// What creation.py:312-379 does with a node whose cells are sorted into buckets.  count(b),
// rmin(b), lmax(b): cells and bounds of bucket b (bounds read only where count(b) > 0).  Empty
// buckets are skipped where the reference merges them away (:322-341): only Rmin, Lmax, index and
// size of the non-empty ones matter afterwards.
enum Decision : int { kLeaf = 0, kSplit = 1, kRetry = 2 };

struct Split {
  int decision;
  int plane;      // first bucket on the right
  int left;       // cells on the left
  double Lmax, Rmin;
  bool bad_cost;  // no finite cost
};

template <typename C, typename R, typename L>
__device__ __forceinline__ Split decide(int nb, int size, int att, double range_Rmin, double range_Lmax, C count,
                                        R rmin, L lmax) {
  Split s{kLeaf, -1, 0, -1.0, -1.0, false};
  const double bl = (range_Lmax - range_Rmin) / (double)nb;
  // creation.py:174-213 split_plane: the first strict minimum
  double best = 1.7976931348623157e308, prev_L = 0.0;
  int m = 0;
  long long left = 0;
  for (int b = 0; b < nb; ++b) {
    const int c = count(b);
    if (c == 0) continue;
    if (m > 0) {
      const long long right = (long long)size - left;
      const double left_volume = (prev_L - range_Rmin) / bl;
      const double right_volume = (range_Lmax - rmin(b)) / bl;
      const double cost = left_volume * (double)left + right_volume * (double)right;
      if (cost < best) {
        best = cost;
        s.plane = b;
        s.left = (int)left;
      }
    }
    left += c;
    prev_L = lmax(b);
    ++m;
  }
  if (m == 1) {  // creation.py:343-358: every cell in one bucket
    s.decision = att == 0 ? kRetry : kLeaf;
    return s;
  }
  if (s.plane < 0) {
    s.bad_cost = true;
    return s;
  }
  s.decision = kSplit;
  s.Lmax = -1.7976931348623157e308;
  s.Rmin = 1.7976931348623157e308;
  for (int b = 0; b < nb; ++b) {
    if (count(b) == 0) continue;
    if (b < s.plane) {
      if (lmax(b) > s.Lmax) s.Lmax = lmax(b);
    } else {
      if (rmin(b) < s.Rmin) s.Rmin = rmin(b);
    }
  }
  return s;
}

// ------------------------------------------------------------------- large nodes
// The root: a leaf (n <= cells_per_leaf), a subtree of k_small (n <= T) or the first large node.
// given: the caller's 3 check values and 5 statistics, or null (the statistics are in the header).
__global__ void __launch_bounds__(kBlock) k_init(int n, int cells_per_leaf, int T, const Key* __restrict__ given,
                                                 Work w, int32_t* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    w.perm[0][i] = i;
    out[i] = i;
  }
  const int tiles = (n + kTile - 1) / kTile;
  if (n > T && i < tiles) w.act[0].map[i] = 0;
  if (i == 0) {
    w.cnodes[0] = ct_node{-1.0, -1.0, -1, 0, n, 0};  // creation.py:400-401
    const bool large = n > cells_per_leaf && n > T, small = n > cells_per_leaf && n <= T;
    const Slots& s = w.act[0];
    s.id[0] = 0;
    s.ptr[0] = 0;
    s.size[0] = n;
    s.dim[0] = 0;
    s.att[0] = 0;
    s.depth[0] = 0;
    s.tile0[0] = 0;
    Header& h = *w.head;
    for (int k = 0; k < 3; ++k) h.checks[k] = given ? given[k] : 0;
    if (given)
      for (int k = 0; k < 5; ++k) h.stats[k] = given[3 + k];
    for (int k = 0; k < 4; ++k) s.range[k] = (k & 1) ? h.stats[k] : ~h.stats[k];
    w.small.id[0] = 0;
    w.small.ptr[0] = 0;
    w.small.size[0] = n;
    w.small.dim[0] = 0;
    w.small.depth[0] = 0;
    h.next_id = 1;
    h.err = 0;
    h.depth = 0;
    h.n_small = small ? 1 : 0;
    h.level[0].active = large ? 1 : 0;
    h.level[1].active = 0;
    h.level[0].tiles = large ? tiles : 0;
    h.level[1].tiles = 0;
    h.n_nodes = 0;
    w.group_end[0] = 1;
  }
}

// Buckets of a tile's cells, the tile's bucket counts and the bucket bounds in both dimensions
// (LDS atomics: 16 lanes of a wavefront per address at 4 buckets, a few hundred cycles a tile).
__global__ void __launch_bounds__(kBlock) k_tile_count(int nb, int level, int par, const double* __restrict__ bb,
                                                       Work w) {
  __shared__ int hist[kMaxBuckets];
  __shared__ Key bnd[kMaxBuckets * 4];
  Header* h = w.head;
  const int t = blockIdx.x;
  if (t == 0 && threadIdx.x == 0) {  // k_node_decide of this level fills the next level's lists
    h->level[par ^ 1].active = 0;
    h->level[par ^ 1].tiles = 0;
    w.group_end[level] = h->next_id;
  }
  if (t >= h->level[par].tiles) return;
  const Slots& cur = w.act[par];
  const int s = cur.map[t];
  const int d = cur.dim[s];
  const int begin = (t - cur.tile0[s]) * kTile;
  const int count = min(kTile, cur.size[s] - begin);
  const int base = cur.ptr[s] + begin;
  const double range_Rmin = dval(cur.range[4 * s + 2 * d]);
  const double range_Lmax = dval(cur.range[4 * s + 2 * d + 1]);
  const double bl = (range_Lmax - range_Rmin) / (double)nb;  // creation.py:278
  for (int k = threadIdx.x; k < 4 * nb; k += kBlock) bnd[k] = (k & 1) ? 0ull : ~0ull;
  for (int k = threadIdx.x; k < nb; k += kBlock) hist[k] = 0;
  const int32_t* __restrict__ perm = w.perm[par];
  double4 box[kTileItems];
#pragma unroll
  for (int j = 0; j < kTileItems; ++j) {
    const int p = j * kBlock + threadIdx.x;
    if (p < count) box[j] = ld_box4(bb, perm[base + p]);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kTileItems; ++j) {
    const int p = j * kBlock + threadIdx.x;
    if (p >= count) continue;
    const double4 x = box[j];
    int b = bucket_of(d ? x.z : x.x, d ? x.w : x.y, range_Rmin, bl, nb);
    if (b < 0) {
      h->err = 1;
      b = nb - 1;
    }
    w.bid[base + p] = (uint8_t)b;
    atomicAdd(&hist[b], 1);
    atomicMin(&bnd[4 * b + 0], dkey(x.x));
    atomicMax(&bnd[4 * b + 1], dkey(x.y));
    atomicMin(&bnd[4 * b + 2], dkey(x.z));
    atomicMax(&bnd[4 * b + 3], dkey(x.w));
  }
  __syncthreads();
  for (int k = threadIdx.x; k < 4 * nb; k += kBlock) w.tilebk[(int64_t)t * 4 * nb + k] = bnd[k];
  for (int k = threadIdx.x; k < nb; k += kBlock) w.tilecnt[(int64_t)t * nb + k] = hist[k];
}

// One workgroup per large node.
__global__ void __launch_bounds__(kDecideBlock) k_node_decide(int nb, int cells_per_leaf, int T, int par, Work w) {
  __shared__ Key bnd[kMaxBuckets * 4];
  __shared__ int cnt[kMaxBuckets];
  __shared__ Key lds[kDecideBlock / 64];
  __shared__ int next_slot[2], next_tile[2], next_tiles[2];
  Header* h = w.head;
  const int s = blockIdx.x;
  if (s >= h->level[par].active) return;
  const Slots& cur = w.act[par];
  const Slots& nxt = w.act[par ^ 1];
  const int X = cur.id[s], ptr = cur.ptr[s], size = cur.size[s], dim = cur.dim[s];
  const int att = cur.att[s], depth = cur.depth[s], tile0 = cur.tile0[s];
  auto tiles_of = [](int cells) { return (cells + kTile - 1) / kTile; };
  const int ntiles = tiles_of(size);
  const int tid = threadIdx.x;
  for (int k = tid; k < 4 * nb; k += kDecideBlock) bnd[k] = (k & 1) ? 0ull : ~0ull;
  __syncthreads();
  // bucket bounds over the node's tiles: a lane keeps to one of the 4 nb bounds
  const int keys = 4 * nb, lanes = kDecideBlock / keys * keys;
  if (tid < lanes) {
    const int k = tid % keys;
    Key v = (k & 1) ? 0ull : ~0ull;
    for (int64_t i = tid; i < (int64_t)ntiles * keys; i += lanes) {
      const Key x = w.tilebk[(int64_t)tile0 * keys + i];
      v = (k & 1) ? (x > v ? x : v) : (x < v ? x : v);
    }
    if (k & 1) atomicMax(&bnd[k], v);
    else atomicMin(&bnd[k], v);
  }
  // prefix of the tile counts, two buckets per scan (a node has fewer than 2^30 cells)
  for (int b = 0; b < nb; b += 2) {
    const bool two = b + 1 < nb;
    Key carry = 0;
    for (int t0 = 0; t0 < ntiles; t0 += kDecideBlock) {
      const int t = t0 + tid;
      const int64_t at = (int64_t)(tile0 + t) * nb + b;
      Key v = 0;
      if (t < ntiles) v = (Key)(unsigned)w.tilecnt[at] | (two ? (Key)(unsigned)w.tilecnt[at + 1] << 32 : 0ull);
      Key total;
      const Key e = carry + block_exclusive_scan<Key, kDecideBlock>(v, lds, &total);
      if (t < ntiles) {
        w.tilepre[at] = (int)(unsigned)e;
        if (two) w.tilepre[at + 1] = (int)(unsigned)(e >> 32);
      }
      carry += total;
    }
    if (tid == 0) {
      cnt[b] = (int)(unsigned)carry;
      if (two) cnt[b + 1] = (int)(unsigned)(carry >> 32);
    }
  }
  __syncthreads();
  if (tid == 0) {
    next_slot[0] = next_slot[1] = -1;
    int off = ptr;
    for (int b = 0; b < nb; ++b) {
      w.boff[s * nb + b] = off;
      off += cnt[b];
    }
    const Key* range = cur.range + 4 * s;
    const double range_Rmin = dval(range[2 * dim]), range_Lmax = dval(range[2 * dim + 1]);
    const Split sp = decide(
        nb, size, att, range_Rmin, range_Lmax, [&](int b) { return cnt[b]; },
        [&](int b) { return dval(bnd[4 * b + 2 * dim]); }, [&](int b) { return dval(bnd[4 * b + 2 * dim + 1]); });
    const int ndim = dim ? 0 : 1;
    auto push_large = [&](int which, int ns, int t0, int id, int cptr, int csize, int catt, int cdepth, const Key (&r)[4]) {
      nxt.id[ns] = id;
      nxt.ptr[ns] = cptr;
      nxt.size[ns] = csize;
      nxt.dim[ns] = ndim;
      nxt.att[ns] = catt;
      nxt.depth[ns] = cdepth;
      nxt.tile0[ns] = t0;
      for (int k = 0; k < 4; ++k) nxt.range[4 * ns + k] = r[k];
      next_slot[which] = ns;
      next_tile[which] = t0;
      next_tiles[which] = tiles_of(csize);
    };
    // two counters that lie together, the first in the low half
    auto raise = [](int32_t* first, int a, int b) {
      return atomicAdd(reinterpret_cast<Key*>(first), (Key)(unsigned)a | (Key)(unsigned)b << 32);
    };
    int32_t* const level = &h->level[par ^ 1].active;
    if (sp.bad_cost) h->err = 2;
    if (sp.decision == kRetry) {
      w.cnodes[X].dim = ndim;
      const Key r[4] = {range[0], range[1], range[2], range[3]};
      const Key at = raise(level, 1, ntiles);
      push_large(0, (int)(unsigned)at, (int)(at >> 32), X, ptr, size, 1, depth, r);
    } else if (sp.decision == kSplit) {
      const int csizes[2] = {sp.left, size - sp.left};
      int smalls = 0, larges = 0, tiles = 0;
      for (int side = 0; side < 2; ++side) {
        if (csizes[side] <= cells_per_leaf) continue;
        if (csizes[side] <= T) {
          ++smalls;
        } else {
          ++larges;
          tiles += tiles_of(csizes[side]);
        }
      }
      const Key ids = raise(&h->next_id, 2, smalls);
      Key at = larges ? raise(level, larges, tiles) : 0;
      const int c = (int)(unsigned)ids;
      int small = (int)(ids >> 32);
      w.cnodes[X].Lmax = sp.Lmax;
      w.cnodes[X].Rmin = sp.Rmin;
      w.cnodes[X].child = c;
      if (h->depth < depth + 1) atomicMax(&h->depth, depth + 1);
      for (int side = 0; side < 2; ++side) {
        const int id = c + side, cptr = side ? ptr + sp.left : ptr, csize = csizes[side];
        w.cnodes[id] = ct_node{-1.0, -1.0, -1, cptr, csize, ndim};  // creation.py:27-29
        if (csize <= cells_per_leaf) continue;
        if (csize <= T) {
          const int k = small++;
          w.small.id[k] = id;
          w.small.ptr[k] = cptr;
          w.small.size[k] = csize;
          w.small.dim[k] = ndim;
          w.small.depth[k] = depth + 1;
          continue;
        }
        Key r[4] = {~0ull, 0ull, ~0ull, 0ull};
        for (int b = side ? sp.plane : 0; b < (side ? nb : sp.plane); ++b)
          for (int k = 0; k < 4; ++k) {
            const Key x = bnd[4 * b + k];  // the neutral key for an empty bucket
            r[k] = (k & 1) ? (x > r[k] ? x : r[k]) : (x < r[k] ? x : r[k]);
          }
        push_large(side, (int)(unsigned)at, (int)(at >> 32), id, cptr, csize, 0, depth + 1, r);
        at += (Key)1 | (Key)(unsigned)tiles_of(csize) << 32;
      }
    }
  }
  __syncthreads();
  for (int k = 0; k < 2; ++k)
    if (next_slot[k] >= 0)
      for (int t = tid; t < next_tiles[k]; t += kDecideBlock) nxt.map[next_tile[k] + t] = next_slot[k];
}

// Bucket counts packed 16 bits each, four to a word: prefix and per-node totals of all buckets
// of a tile (or a subtree's level) in one scan a word.
__device__ __forceinline__ int packed(Key w, int b) { return (int)((w >> (16 * (b & 3))) & 0xffffu); }

// The cells of a tile to their buckets, in order.  `out` always holds the latest order of every
// position, whichever level a position is last touched at.
__global__ void __launch_bounds__(kBlock) k_tile_scatter(int nb, int par, Work w, int32_t* __restrict__ out) {
  __shared__ Key lds[kBlock / 64];
  const int t = blockIdx.x;
  if (t >= w.head->level[par].tiles) return;
  const Slots& cur = w.act[par];
  const int s = cur.map[t];
  const int begin = (t - cur.tile0[s]) * kTile;
  const int count = min(kTile, cur.size[s] - begin);
  const int base = cur.ptr[s] + begin;
  int c[kTileItems], b[kTileItems];
#pragma unroll
  for (int j = 0; j < kTileItems; ++j) {
    const int p = threadIdx.x * kTileItems + j;
    c[j] = p < count ? w.perm[par][base + p] : -1;
    b[j] = p < count ? (int)w.bid[base + p] : -4;
  }
  for (int word = 0; word < (nb + 3) / 4; ++word) {
    Key v = 0;
#pragma unroll
    for (int j = 0; j < kTileItems; ++j)
      if ((b[j] >> 2) == word) v += 1ull << (16 * (b[j] & 3));
    Key total;
    Key run = block_exclusive_scan<Key>(v, lds, &total);
#pragma unroll
    for (int j = 0; j < kTileItems; ++j) {
      if ((b[j] >> 2) != word) continue;
      const int q = w.boff[s * nb + b[j]] + w.tilepre[(int64_t)t * nb + b[j]] + packed(run, b[j]);
      w.perm[par ^ 1][q] = c[j];
      out[q] = c[j];
      run += 1ull << (16 * (b[j] & 3));
    }
  }
}

// ------------------------------------------------------------------- subtrees in LDS
__device__ __forceinline__ double4 box_union(double4 a, double4 b) {  // NaN poisons the union
  const double nan = __builtin_nan("");
  const bool bad = isnan(a.x) || isnan(a.y) || isnan(a.z) || isnan(a.w) || isnan(b.x) || isnan(b.y) ||
                   isnan(b.z) || isnan(b.w);
  if (bad) return make_double4(nan, nan, nan, nan);
  return make_double4(b.x < a.x ? b.x : a.x, b.y > a.y ? b.y : a.y, b.z < a.z ? b.z : a.z,
                      b.w > a.w ? b.w : a.w);
}

__device__ __forceinline__ double4 empty_box() {
  const double inf = __builtin_inf();
  return make_double4(inf, -inf, inf, -inf);
}

// One workgroup builds the whole subtree of a node of at most T cells: the levels of creation.py
// run one after the other over the subtree's positions, T / THREADS of them per lane, with LDS
// arrays and barriers where the large nodes have global arrays and kernels.  A cell's box is
// gathered (16 bytes of it) once per level; everything else is in LDS.
//   per level:  1 extents per node (a wavefront whose positions share one node reduces in
//                 registers; otherwise LDS atomics)
//               2 buckets, and the prefix over positions of the packed bucket counts
//               3 the cells to their buckets; bucket bounds (LDS atomics)
//               4 split decisions, one lane per node
//               5 positions to the children's slots
// NB: the bucket class (>= nb).
template <int NB, int T, int THREADS>
__global__ void __launch_bounds__(THREADS) k_small(int nb, int cells_per_leaf, int first, int want_boxes,
                                                   const double* __restrict__ bb, Work w, int32_t* out) {
  constexpr int IT = T / THREADS;
  constexpr int W = NB / 4;
  constexpr int S = T / 2;  // an active node has at least two cells
  static_assert(T <= 1024 && IT * THREADS == T, "16-bit packed counts and node ids");
  __shared__ int perm[T];
  __shared__ short seg[T];
  __shared__ Key pre[W][T + 1];
  __shared__ Key rmin[S], rmax[S];
  __shared__ Key bnd[2][S * NB];
  __shared__ uint16_t sptr[2][S], ssize[2][S], sid[2][S], sdepth[2][S];
  __shared__ uint8_t sdim[2][S], satt[2][S];
  __shared__ uint16_t dright[S];
  __shared__ short dl[S], dr[S];
  __shared__ uint16_t child[2 * T];
  __shared__ uint16_t gend[2 * T + 4];
  __shared__ Key wave_tot[W][THREADS / 64];
  __shared__ int next_id, n_next, max_depth, err;
  // after the last level: node counts and ranks, where the bucket bounds were
  uint16_t* ic = reinterpret_cast<uint16_t*>(&bnd[0][0]);
  uint16_t* rk = ic + 2 * T;
  uint16_t* li = rk + 2 * T;
  static_assert(sizeof(bnd) >= 3 * 2 * T * sizeof(uint16_t), "node arrays fit the bucket bounds");
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;

  for (int si = first + blockIdx.x; si < w.head->n_small; si += gridDim.x) {
    const int root = w.small.id[si], base = w.small.ptr[si], m = w.small.size[si];
    ct_node* ln = w.lnodes + 2 * (int64_t)base;
    double4* lb = w.lbox + 2 * (int64_t)base;
    auto node = [&](int x) { return x == 0 ? w.cnodes + root : ln + x; };
    __syncthreads();  // the previous subtree's arrays are done with
    for (int p = tid; p < T; p += THREADS) {
      perm[p] = p < m ? out[base + p] : -1;
      seg[p] = p < m ? 0 : -1;
    }
    if (tid == 0) {
      sptr[0][0] = 0;
      ssize[0][0] = (uint16_t)m;
      sid[0][0] = 0;
      sdepth[0][0] = 0;
      sdim[0][0] = (uint8_t)w.small.dim[si];
      satt[0][0] = 0;
      next_id = 1;
      n_next = 0;
      max_depth = 0;
      err = 0;
      gend[0] = 1;
      child[0] = 0;
      rmin[0] = ~0ull;
      rmax[0] = 0ull;
    }
    for (int k = tid; k < NB; k += THREADS) {
      bnd[0][k] = ~0ull;
      bnd[1][k] = 0ull;
    }
    int A = 1, cur = 0, G = 0;
    __syncthreads();
    while (A > 0) {
      // 1: extents
      int c[IT], s[IT];
      Key lo[IT], hi[IT];
#pragma unroll
      for (int j = 0; j < IT; ++j) {
        const int p = tid * IT + j;
        s[j] = seg[p];
        c[j] = perm[p];
        lo[j] = ~0ull;
        hi[j] = 0ull;
        if (s[j] >= 0) {
          const double2 x = reinterpret_cast<const double2*>(bb)[2 * (int64_t)c[j] + sdim[cur][s[j]]];
          lo[j] = dkey(x.x);
          hi[j] = dkey(x.y);
        }
      }
      {
        bool one = true;
        const int s0 = __builtin_amdgcn_readfirstlane(s[0]);
        Key l = lo[0], h = hi[0];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
          one = one && s[j] == s0;
          l = lo[j] < l ? lo[j] : l;
          h = hi[j] > h ? hi[j] : h;
        }
        if (__all(one)) {
          if (s0 >= 0) {
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
              const Key l2 = __shfl_xor(l, d, 64), h2 = __shfl_xor(h, d, 64);
              l = l2 < l ? l2 : l;
              h = h2 > h ? h2 : h;
            }
            if (lane == 0) {
              atomicMin(&rmin[s0], l);
              atomicMax(&rmax[s0], h);
            }
          }
        } else {
#pragma unroll
          for (int j = 0; j < IT; ++j) {
            if (s[j] < 0) continue;
            atomicMin(&rmin[s[j]], lo[j]);
            atomicMax(&rmax[s[j]], hi[j]);
          }
        }
      }
      __syncthreads();
      // 2: buckets and the prefix of their packed counts
      int b[IT];
      Key mine[W], incl[W];
#pragma unroll
      for (int k = 0; k < W; ++k) mine[k] = 0;
#pragma unroll
      for (int j = 0; j < IT; ++j) {
        b[j] = -4;
        if (s[j] < 0) continue;
        const double range_Rmin = dval(rmin[s[j]]);
        const double bl = (dval(rmax[s[j]]) - range_Rmin) / (double)nb;
        b[j] = bucket_of(dval(lo[j]), dval(hi[j]), range_Rmin, bl, nb);
        if (b[j] < 0) {
          err = 1;
          b[j] = nb - 1;
        }
#pragma unroll
        for (int k = 0; k < W; ++k)
          if ((b[j] >> 2) == k) mine[k] += 1ull << (16 * (b[j] & 3));
      }
#pragma unroll
      for (int k = 0; k < W; ++k) {
        Key x = mine[k];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const Key y = __shfl_up(x, d, 64);
          if (lane >= d) x += y;
        }
        incl[k] = x;
        if (lane == 63) wave_tot[k][wave] = x;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < W; ++k) {
        Key run = incl[k] - mine[k];
        for (int v = 0; v < THREADS / 64; ++v)
          if (v < wave) run += wave_tot[k][v];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
          pre[k][tid * IT + j] = run;
          if ((b[j] >> 2) == k) run += 1ull << (16 * (b[j] & 3));
        }
        if (tid == THREADS - 1) pre[k][T] = run;
      }
      __syncthreads();
      // 3: the cells to their buckets
#pragma unroll
      for (int j = 0; j < IT; ++j) {
        if (s[j] < 0) continue;
        const int p = tid * IT + j, sl = s[j];
        const int a = sptr[cur][sl], e = a + ssize[cur][sl];
        int q = a;
#pragma unroll
        for (int k = 0; k < W; ++k) {
          const Key p0 = pre[k][a], tot = pre[k][e] - p0;
#pragma unroll
          for (int f = 0; f < 4; ++f)
            if (4 * k + f < b[j]) q += packed(tot, f);
          if ((b[j] >> 2) == k) q += packed(pre[k][p] - p0, b[j]);
        }
        perm[q] = c[j];
        atomicMin(&bnd[0][sl * NB + b[j]], lo[j]);
        atomicMax(&bnd[1][sl * NB + b[j]], hi[j]);
      }
      __syncthreads();
      // 4: decisions
      const int nx = cur ^ 1;
      for (int sl = tid; sl < A; sl += THREADS) {
        const int a = sptr[cur][sl], size = ssize[cur][sl], X = sid[cur][sl], dim = sdim[cur][sl];
        const int depth = sdepth[cur][sl], ndim = dim ? 0 : 1;
        const double range_Rmin = dval(rmin[sl]), range_Lmax = dval(rmax[sl]);
        auto push = [&](int id, int cptr, int csize, int catt, int cdepth) -> int {
          const int ns = atomicAdd(&n_next, 1);
          sptr[nx][ns] = (uint16_t)cptr;
          ssize[nx][ns] = (uint16_t)csize;
          sid[nx][ns] = (uint16_t)id;
          sdim[nx][ns] = (uint8_t)ndim;
          satt[nx][ns] = (uint8_t)catt;
          sdepth[nx][ns] = (uint16_t)cdepth;
          return ns;
        };
        auto split = [&](double Lmax, double Rmin, int left) {
          ct_node* nd = node(X);
          const int ch = atomicAdd(&next_id, 2);
          nd->Lmax = Lmax;
          nd->Rmin = Rmin;
          nd->child = X == 0 ? -2 : 1;  // linked by k_emit
          child[X] = (uint16_t)ch;
          child[ch] = child[ch + 1] = 0;
          ln[ch] = ct_node{-1.0, -1.0, -1, base + a, left, ndim};  // creation.py:27-29
          ln[ch + 1] = ct_node{-1.0, -1.0, -1, base + a + left, size - left, ndim};
          dright[sl] = (uint16_t)(a + left);
          dl[sl] = left > cells_per_leaf ? (short)push(ch, a, left, 0, depth + 1) : (short)-1;
          dr[sl] = size - left > cells_per_leaf ? (short)push(ch + 1, a + left, size - left, 0, depth + 1) : (short)-1;
          atomicMax(&max_depth, depth + 1);
        };
        dright[sl] = 0;
        dl[sl] = dr[sl] = -1;
        if (cells_per_leaf == 1 && size == 2) {  // creation.py:312-320
          split(range_Lmax, range_Rmin, 1);
          continue;
        }
        Key tot[W];
#pragma unroll
        for (int k = 0; k < W; ++k) tot[k] = pre[k][a + size] - pre[k][a];
        const Split sp = decide(
            nb, size, satt[cur][sl], range_Rmin, range_Lmax,
            [&](int k) {
              Key x = tot[0];
#pragma unroll
              for (int v = 1; v < W; ++v) x = (k >> 2) == v ? tot[v] : x;
              return packed(x, k);
            },
            [&](int k) { return dval(bnd[0][sl * NB + k]); }, [&](int k) { return dval(bnd[1][sl * NB + k]); });
        if (sp.bad_cost) err = 2;
        if (sp.decision == kRetry) {
          node(X)->dim = ndim;
          dl[sl] = dr[sl] = (short)push(X, a, size, 1, depth);
        } else if (sp.decision == kSplit) {
          split(sp.Lmax, sp.Rmin, sp.left);
        }
      }
      __syncthreads();
      // 5: positions to their children's slots; the next level's reduction targets
      const int An = n_next;
#pragma unroll
      for (int j = 0; j < IT; ++j) {
        if (s[j] < 0) continue;
        const int p = tid * IT + j;
        seg[p] = p < (int)dright[s[j]] ? dl[s[j]] : dr[s[j]];
      }
      for (int k = tid; k < An; k += THREADS) {
        rmin[k] = ~0ull;
        rmax[k] = 0ull;
      }
      for (int k = tid; k < An * NB; k += THREADS) {
        bnd[0][k] = ~0ull;
        bnd[1][k] = 0ull;
      }
      __syncthreads();
      ++G;
      if (tid == 0) {
        n_next = 0;
        gend[G] = (uint16_t)next_id;
      }
      A = An;
      cur = nx;
    }
    __syncthreads();
    const int N = next_id;
    for (int p = tid; p < m; p += THREADS) out[base + p] = perm[p];
    // leaves, then internal nodes bottom-up: internal nodes per subtree, tight boxes
    for (int x = tid; x < N; x += THREADS) {
      if (child[x] != 0) continue;
      ic[x] = 0;
      if (!want_boxes) continue;
      const ct_node nd = *node(x);
      double4 u = empty_box();
      for (int k = nd.ptr - base; k < nd.ptr - base + nd.size; ++k) u = box_union(u, ld_box4(bb, perm[k]));
      (x == 0 ? w.tbox[root] : lb[x]) = u;
    }
    __syncthreads();
    for (int g = G; g >= 0; --g) {
      const int lo = g == 0 ? 0 : gend[g - 1], hi = gend[g];
      for (int x = lo + tid; x < hi; x += THREADS) {
        const int ch = child[x];
        if (ch == 0) continue;
        ic[x] = (uint16_t)(1 + ic[ch] + ic[ch + 1]);
        if (want_boxes) (x == 0 ? w.tbox[root] : lb[x]) = box_union(lb[ch], lb[ch + 1]);
      }
      __syncthreads();
    }
    // top-down: ranks and DFS indices
    if (tid == 0) {
      rk[0] = 0;
      li[0] = 0;
    }
    __syncthreads();
    for (int g = 0; g <= G; ++g) {
      const int lo = g == 0 ? 0 : gend[g - 1], hi = gend[g];
      for (int x = lo + tid; x < hi; x += THREADS) {
        const int ch = child[x];
        if (ch == 0) continue;
        const int r = rk[x];
        li[ch] = (uint16_t)(1 + 2 * r);
        li[ch + 1] = (uint16_t)(2 + 2 * r);
        rk[ch] = (uint16_t)(r + 1);
        rk[ch + 1] = (uint16_t)(r + 1 + ic[ch]);
      }
      __syncthreads();
    }
    for (int x = tid; x < N; x += THREADS)
      if (x > 0) w.lmeta[2 * (int64_t)base + x] = (int)((unsigned)li[x] | ((unsigned)rk[x] << 16));
    if (tid == 0) {
      w.icount[root] = ic[0];
      atomicMax(&w.head->depth, w.small.depth[si] + max_depth);
      if (err) w.head->err = err;
    }
  }
}

// ------------------------------------------------------------------- numbering
// The large-node stage's nodes: internal nodes per subtree and tight boxes bottom-up, DFS ranks
// top-down, by creation level.  There are about 2 n / T of them, so one workgroup does it.
constexpr int kTopBlock = 1024;
constexpr int kTopLevels = 64;  // batches of levels that end by here run k_top before they are read back

__global__ void __launch_bounds__(kTopBlock) k_top(int levels, int want_boxes, const double* __restrict__ bb, Work w,
                                                   const int32_t* __restrict__ cells) {
  const int tid = threadIdx.x, M = w.head->next_id;
  ct_node* cn = w.cnodes;
  // Leaves, found 64 nodes at a time (a node at a time, 3000 nodes of 999,941 cells took 50 of the
  // kernel's 61 us), then a wavefront each.
  for (int x0 = tid & ~63; x0 < M; x0 += kTopBlock) {
    const int mine = x0 + lane_id();
    for (uint64_t todo = __ballot(mine < M && cn[mine < M ? mine : 0].child == -1); todo; todo &= todo - 1) {
      const int x = x0 + __ffsll((unsigned long long)todo) - 1;
      const ct_node nd = cn[x];
      double4 u = empty_box();
      if (want_boxes) {
        for (int k = nd.ptr + lane_id(); k < nd.ptr + nd.size; k += 64) u = box_union(u, ld_box4(bb, cells[k]));
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
          const double4 v = make_double4(__shfl_xor(u.x, d, 64), __shfl_xor(u.y, d, 64), __shfl_xor(u.z, d, 64),
                                         __shfl_xor(u.w, d, 64));
          u = box_union(u, v);
        }
      }
      if (lane_id() == 0) {
        w.icount[x] = 0;
        if (want_boxes) w.tbox[x] = u;
      }
    }
  }
  __syncthreads();
  for (int g = levels; g >= 0; --g) {
    const int lo = g == 0 ? 0 : w.group_end[g - 1], hi = g == levels ? M : w.group_end[g];
    for (int x = lo + tid; x < hi; x += kTopBlock) {
      const int c = cn[x].child;
      if (c < 0) continue;
      w.icount[x] = 1 + w.icount[c] + w.icount[c + 1];
      if (want_boxes) w.tbox[x] = box_union(w.tbox[c], w.tbox[c + 1]);
    }
    __syncthreads();
  }
  if (tid == 0) {
    w.drank[0] = 0;
    w.newidx[0] = 0;
  }
  __syncthreads();
  for (int g = 0; g <= levels; ++g) {
    const int lo = g == 0 ? 0 : w.group_end[g - 1], hi = g == levels ? M : w.group_end[g];
    for (int x = lo + tid; x < hi; x += kTopBlock) {
      const int c = cn[x].child;
      if (c < 0) continue;
      const int r = w.drank[x];
      w.newidx[c] = 1 + 2 * r;
      w.newidx[c + 1] = 2 + 2 * r;
      w.drank[c] = r + 1;
      w.drank[c + 1] = r + 1 + w.icount[c];
    }
    __syncthreads();
  }
  if (tid == 0) w.head->n_nodes = 1 + 2 * w.icount[0];
}

// Nodes to their reference indices: workgroups below n_small copy a subtree each (its nodes are
// 2 r + 1 ... 2 r + 2 * internal), the others the large-node stage's nodes.
__global__ void __launch_bounds__(kBlock) k_emit(int n_small, int n_top, Work w, ct_node* __restrict__ nodes,
                                                 double4* __restrict__ boxes) {
  if ((int)blockIdx.x < n_small) {
    const int root = w.small.id[blockIdx.x];
    const int64_t at = 2 * (int64_t)w.small.ptr[blockIdx.x];
    const int r = w.drank[root], count = 2 * w.icount[root];
    for (int x = 1 + threadIdx.x; x <= count; x += kBlock) {
      const unsigned meta = (unsigned)w.lmeta[at + x];
      ct_node nd = w.lnodes[at + x];
      nd.child = nd.child >= 0 ? 1 + 2 * (r + (int)(meta >> 16)) : -1;
      const int64_t i = 2 * (int64_t)r + (meta & 0xffffu);
      nodes[i] = nd;
      if (boxes) boxes[i + 1] = w.lbox[at + x];
    }
    return;
  }
  const int x = ((int)blockIdx.x - n_small) * kBlock + threadIdx.x;
  if (x == 0 && boxes) {
    const double nan = __builtin_nan("");
    boxes[0] = make_double4(nan, nan, nan, nan);  // row 0 is not a node's
  }
  if (x >= n_top) return;
  ct_node nd = w.cnodes[x];
  nd.child = nd.child == -1 ? -1 : 1 + 2 * w.drank[x];
  nodes[w.newidx[x]] = nd;
  if (boxes) boxes[w.newidx[x] + 1] = w.tbox[x];
}

// A lane per cell while there are no more subtrees than CUs (about 2 n / T of them), two cells per lane
// and two workgroups a CU above: 20,000 cells 315 instead of 344 us, 999,941 cells 1283 against 1136.
constexpr int64_t kWideCells = 128 * 1024;

int launch_small(int64_t n, int nb, int cells_per_leaf, int first, int want_boxes, const double* bb, const Work& w,
                 int32_t* out, unsigned grid, hipStream_t st) {
  const bool wide = n <= kWideCells;
  if (nb <= 4 && wide) k_small<4, 1024, 1024><<<grid, 1024, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  else if (nb <= 8 && wide) k_small<8, 1024, 1024><<<grid, 1024, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  else if (nb <= 4) k_small<4, 1024, 512><<<grid, 512, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  else if (nb <= 8) k_small<8, 1024, 512><<<grid, 512, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  else if (nb <= 16) k_small<16, 512, 256><<<grid, 256, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  else if (nb <= 32) k_small<32, 256, 256><<<grid, 256, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  else k_small<64, 128, 128><<<grid, 128, 0, st>>>(nb, cells_per_leaf, first, want_boxes, bb, w, out);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int check_build(int64_t n, int32_t nb, int32_t cpl, size_t workspace_bytes) {
  CT_REQUIRE(n >= 1 && n < (int64_t)1 << 30, "n_elements must be in [1, 2^30)");
  CT_REQUIRE(nb >= 2 && nb <= kMaxBuckets, "n_buckets must be in [2, %d]", kMaxBuckets);
  CT_REQUIRE(cpl >= 1, "cells_per_leaf must be >= 1");
  size_t need = 0;
  carve(nullptr, n, nb, &need);
  if (workspace_bytes < need) {
    set_error("build workspace too small: %zu < %zu", workspace_bytes, need);
    return CT_ERR_WORKSPACE;
  }
  return CT_OK;
}

}  // namespace
}  // namespace ct

using namespace ct;

extern "C" {

int ct_check_values(const uint64_t* checks_host, int64_t* out3_host) {
  CT_REQUIRE(checks_host && out3_host, "null pointer");
  for (int k = 0; k < 3; ++k) out3_host[k] = (int64_t)((k ? ~checks_host[k] : checks_host[k]) ^ 0x8000000000000000ull);
  return CT_OK;
}

int64_t ct_max_nodes(int64_t n_elements) {  // creation.py:216-230
  int64_t n_nodes = n_elements;
  int64_t nodes = (n_elements + 1) / 2;
  while (nodes > 1) {
    n_nodes += nodes;
    nodes = (nodes + 1) / 2;
  }
  return n_nodes + 1;
}

size_t ct_build_workspace_bytes(int64_t n_elements, int32_t n_buckets) {
  size_t total = 0;
  const int nb = n_buckets < 2 ? 2 : (n_buckets > kMaxBuckets ? kMaxBuckets : n_buckets);
  carve(nullptr, n_elements < 1 ? 1 : n_elements, nb, &total);
  return total;
}

int ct_build_plan(const double* bb_coords, int64_t n_elements, int32_t n_buckets, int32_t cells_per_leaf,
                  int32_t want_boxes, void* workspace, size_t workspace_bytes, int32_t* bb_indices_out,
                  double* distances, const uint64_t* checks, ct_build_info* info, void* stream) {
  int rc = check_build(n_elements, n_buckets, cells_per_leaf, workspace_bytes);
  if (rc) return rc;
  CT_REQUIRE(workspace && bb_indices_out && bb_coords && info, "null pointer");
  hipStream_t st = as_stream(stream);
  size_t need = 0;
  const Work w = carve(static_cast<char*>(workspace), n_elements, n_buckets, &need);
  const int n = (int)n_elements, nb = n_buckets, cpl = cells_per_leaf, T = small_cells(nb);

  if (checks == nullptr) {
    rc = bbox_stat_keys(bb_coords, n, distances, w.head->stats, st);
    if (rc) return rc;
  }
  k_init<<<grid_for(n), kBlock, 0, st>>>(n, cpl, T, reinterpret_cast<const Key*>(checks), w, bb_indices_out);
  CT_LAUNCH_CHECK();

  Header h{};
  auto read_header = [&]() -> int {
    CT_HIP(hipMemcpyAsync(&h, w.head, sizeof(h), hipMemcpyDeviceToHost, st));
    CT_HIP(hipStreamSynchronize(st));
    return CT_OK;
  };
  int levels = 0, done_small = 0;
  // levels of a balanced tree above the subtrees, plus two; then more, in growing batches
  int batch = 0;
  if (n > T && n > cpl) {
    batch = 2;
    for (int64_t m = T; m < n; m *= 2) ++batch;
  }
  while (true) {
    for (int k = 0; k < batch; ++k, ++levels) {
      const int par = levels & 1;
      const int64_t active = levels < 30 ? std::min((int64_t)1 << levels, max_active(n, nb)) : max_active(n, nb);
      const unsigned tiles = (unsigned)std::min((int64_t)n / kTile + active + 1, max_tiles(n, nb));
      k_tile_count<<<tiles, kBlock, 0, st>>>(nb, levels, par, bb_coords, w);
      CT_LAUNCH_CHECK();
      k_node_decide<<<(unsigned)active, kDecideBlock, 0, st>>>(nb, cpl, T, par, w);
      CT_LAUNCH_CHECK();
      k_tile_scatter<<<tiles, kBlock, 0, st>>>(nb, par, w, bb_indices_out);
      CT_LAUNCH_CHECK();
    }
    const unsigned small_grid = (unsigned)std::min((int64_t)2048, (int64_t)n / 2 + 1);
    rc = launch_small(n, nb, cpl, done_small, want_boxes, bb_coords, w, bb_indices_out, small_grid, st);
    if (rc) return rc;
    // k_top goes along where this batch may be the last; it passes over all levels, so a deep chain
    // runs it once, at the end (a fan of 200,000 triangles, 19,081 levels: 1.0 s, and 25.3 with one a batch).
    const bool topped = levels <= kTopLevels;
    if (topped) {
      k_top<<<1, kTopBlock, 0, st>>>(levels, want_boxes, bb_coords, w, bb_indices_out);
      CT_LAUNCH_CHECK();
    }
    rc = read_header();
    if (rc) return rc;
    done_small = h.n_small;
    if (h.err != 0) break;
    if (h.level[levels & 1].active == 0) {
      if (topped) break;
      k_top<<<1, kTopBlock, 0, st>>>(levels, want_boxes, bb_coords, w, bb_indices_out);
      CT_LAUNCH_CHECK();
      rc = read_header();
      if (rc) return rc;
      break;
    }
    // Children are strictly smaller than their parent and a node retries once, so the loop
    // ends within 2 * n_elements levels (the length of group_end); the guard only protects it.
    batch = std::min(std::max(2 * batch, 8), 64);
    if (levels + batch > 2 * (int64_t)n + 4) batch = (int)(2 * (int64_t)n + 4 - levels);
    if (batch <= 0) {
      set_error("tree build did not converge");
      return CT_ERR_DEGENERATE;
    }
  }
  info->n_nodes = h.n_nodes;
  info->depth = h.depth;
  info->n_top = h.next_id;
  info->n_small = h.n_small;
  info->reserved = 0;
  for (int k = 0; k < 5; ++k) info->stats[k] = dval((k == 0 || k == 2) ? ~h.stats[k] : h.stats[k]);
  ct_check_values(reinterpret_cast<const uint64_t*>(h.checks), info->checks);
  if (checks == nullptr)
    for (int64_t& c : info->checks) c = 0;
  if (h.err != 0) {
    set_error(h.err == 1 ? "degenerate bucketing: a cell centroid falls outside every bucket"
                         : "degenerate bucketing: no finite split cost");
    return CT_ERR_DEGENERATE;
  }
  return CT_OK;
}

int ct_build_emit(int64_t n_elements, int32_t n_buckets, void* workspace, size_t workspace_bytes,
                  const ct_build_info* info, ct_node* nodes_out, double* node_boxes_out, void* stream) {
  int rc = check_build(n_elements, n_buckets, 1, workspace_bytes);
  if (rc) return rc;
  CT_REQUIRE(workspace && info && nodes_out && info->n_top >= 1 && info->n_small >= 0, "bad arguments");
  size_t need = 0;
  const Work w = carve(static_cast<char*>(workspace), n_elements, n_buckets, &need);
  k_emit<<<(unsigned)info->n_small + grid_for(info->n_top), kBlock, 0, as_stream(stream)>>>(
      info->n_small, info->n_top, w, nodes_out, reinterpret_cast<double4*>(node_boxes_out));
  CT_LAUNCH_CHECK();
  return CT_OK;
}

int ct_build(const double* bb_coords, int64_t n_elements, int32_t n_buckets, int32_t cells_per_leaf,
             void* workspace, size_t workspace_bytes, ct_node* nodes_out, int32_t* bb_indices_out,
             int64_t* n_nodes, int32_t* depth, void* stream) {
  CT_REQUIRE(n_nodes && depth && nodes_out, "null pointer");
  ct_build_info info{};
  int rc = ct_build_plan(bb_coords, n_elements, n_buckets, cells_per_leaf, 0, workspace, workspace_bytes,
                         bb_indices_out, nullptr, nullptr, &info, stream);
  if (rc) return rc;
  rc = ct_build_emit(n_elements, n_buckets, workspace, workspace_bytes, &info, nodes_out, nullptr, stream);
  if (rc) return rc;
  *n_nodes = info.n_nodes;
  *depth = info.depth;
  return CT_OK;
}

}  // extern "C"
