// ct_lists.hip -- the lists a regridding gathers through: the pairs of every source cell, the face
// corners of every vertex of both meshes, and the first pair of every target.
//
// All three groupings ("the items of every key, ascending") are made together, in one key space
// (source cells, target vertices, source vertices) over one item space (pairs, target corners, source
// corners): counts by atomics, a scan, the items of a key in arrival order, then every item's rank
// among its key's.  Most keys have 2 to 10 items, so an item finds its rank by comparing with the
// others (kCompare at most); longer lists are sorted by a wavefront in registers, still longer ones by
// a workgroup.  Bound by the atomics and by launches: 9 kernels and no synchronization instead of
// stable sorts, histograms and selections by a library (190 kernels and 12 synchronizations, 1.0 of
// the 1.69 ms of a setup with 180,000 source cells and 61,009 targets; now 0.15 of 0.51).
#include <algorithm>

#include "ct_internal.h"
#include "ct_primitives.h"

namespace ct {
namespace {

constexpr int kGroups = 3;  // pairs by source, target corners by vertex, source corners by vertex
constexpr int kCompare = 64;
constexpr int kWaveMax = 1024;
constexpr int kHugeBlock = 1024;
constexpr int kHugeLds = 8192;  // items sorted in LDS; longer lists stream over all items
constexpr int kHugeStream = 8;  // items a lane takes at a time then

constexpr uint32_t kNone = ~0u;
constexpr int64_t kItemsPerLaunch = (int64_t)1 << 31;  // a HIP launch has fewer than 2^32 lanes

struct Lists {
  const int64_t* ss;
  const int64_t* tt;
  const int32_t* faces[2];    // target, source
  int64_t keys[kGroups + 1];  // first key of every group; all
  int64_t items[kGroups + 1];
  int64_t* offsets[kGroups];  // out: keys + 1 each
  int64_t* list[kGroups];     // out
  int64_t* src_tgt;           // out: the target of every entry of list[0]
  int64_t* counts;            // by key
  int64_t* starts;            // their scan, keys + 1
  uint32_t* unsorted;         // by start: a key's items in arrival order
  uint32_t* rank;             // by item: arrival among its key's, kNone: no key
  uint32_t* longer;           // keys of more than kCompare items
  uint32_t* huge;             // keys of more than kWaveMax
  int32_t* n_longer;          // [0] longer, [1] huge
};

__device__ __forceinline__ int group_of(const int64_t (&first)[kGroups + 1], int64_t x) {
  return (x >= first[1] ? 1 : 0) + (x >= first[2] ? 1 : 0);
}

// The key of item x, -1 for a corner past a face's end.
__device__ __forceinline__ int64_t key_of(const Lists& l, int g, int64_t id) {
  if (g == 0) return l.ss[id];
  const int v = l.faces[g - 1][id];
  return v < 0 ? -1 : l.keys[g] + v;
}

__global__ void __launch_bounds__(kBlock) k_list_count(Lists l, int64_t x0) {
  const int64_t x = x0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
  int64_t key = -1;
  if (x < l.items[kGroups]) {
    const int g = group_of(l.items, x);
    key = key_of(l, g, x - l.items[g]);
  }
  // The lanes with the first lane's key count together (a large cell's pairs follow each other).
  auto* counts = reinterpret_cast<unsigned long long*>(l.counts);
  const int64_t lead = __shfl(key, 0);
  const uint64_t same = __ballot(key == lead);
  const int lane = lane_id();
  uint32_t r = kNone;
  if (lead >= 0 && key == lead) {
    if (lane == 0) r = (uint32_t)atomicAdd(counts + key, (unsigned long long)__popcll(same));
  } else if (key >= 0) {
    r = (uint32_t)atomicAdd(counts + key, 1ull);
  }
  const uint32_t base = __shfl(r, 0);
  if (lead >= 0 && key == lead) r = base + (uint32_t)__popcll(same & ((1ull << lane) - 1));
  if (x < l.items[kGroups]) l.rank[x] = r;
}

__global__ void __launch_bounds__(kBlock) k_list_place(Lists l, int64_t x0) {
  const int64_t x = x0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (x >= l.items[kGroups]) return;
  const uint32_t r = l.rank[x];
  if (r == kNone) return;
  const int g = group_of(l.items, x);
  const int64_t id = x - l.items[g];
  l.unsorted[l.starts[key_of(l, g, id)] + r] = (uint32_t)id;
}

__device__ __forceinline__ void put(const Lists& l, int g, int64_t at, int64_t id) {
  l.list[g][at] = id;
  if (g == 0) l.src_tgt[at] = l.tt[id];
}

// info: [0] rest targets (k_targets), [1] target corners, [2] source corners.
// Offsets of every key, and the place of every item of a key with at most kCompare.
__global__ void __launch_bounds__(kBlock) k_list_rank(Lists l, int64_t x0, int64_t* info) {
  const int64_t x = x0 + (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (x == 0) {
    info[1] = l.starts[l.keys[2]] - l.starts[l.keys[1]];
    info[2] = l.starts[l.keys[3]] - l.starts[l.keys[2]];
  }
  if (x < l.keys[kGroups]) {
    const int g = group_of(l.keys, x);
    const int64_t first = l.starts[l.keys[g]];
    l.offsets[g][x - l.keys[g]] = l.starts[x] - first;
    if (x + 1 == l.keys[g + 1]) l.offsets[g][x + 1 - l.keys[g]] = l.starts[x + 1] - first;
  }
  if (x >= l.items[kGroups]) return;
  const uint32_t arrival = l.rank[x];
  if (arrival == kNone) return;
  const int g = group_of(l.items, x);
  const uint32_t id = (uint32_t)(x - l.items[g]);
  const int64_t key = key_of(l, g, id), b = l.starts[key];
  const int m = (int)(l.starts[key + 1] - b);
  if (m > kCompare) {
    if (arrival == 0) {
      if (m > kWaveMax) l.huge[atomicAdd(l.n_longer + 1, 1)] = (uint32_t)key;
      else l.longer[atomicAdd(l.n_longer, 1)] = (uint32_t)key;
    }
    return;
  }
  int r = 0;
  for (int j = 0; j < m; ++j) r += l.unsorted[b + j] < id ? 1 : 0;
  put(l, g, b - l.starts[l.keys[g]] + r, id);
}

template <int R>
__device__ __forceinline__ void sort_list(const Lists& l, int g, int64_t b, int m, int lane) {
  uint32_t v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = r * 64 + lane < m ? l.unsorted[b + r * 64 + lane] : ~0u;
  wave_sort<R>(v, lane);
  const int64_t at = b - l.starts[l.keys[g]];
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r * 64 + lane < m) put(l, g, at + r * 64 + lane, v[r]);
}

// Keys of kCompare + 1 to kWaveMax items, a wavefront each.
__global__ void __launch_bounds__(kBlock) k_list_longer(Lists l) {
  const int n = l.n_longer[0], lane = lane_id(), waves = gridDim.x * (kBlock / 64);
  for (int i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); i < n; i += waves) {
    const int64_t key = l.longer[i], b = l.starts[key];
    const int m = (int)(l.starts[key + 1] - b), g = group_of(l.keys, key);
    if (m <= 128) sort_list<2>(l, g, b, m, lane);
    else if (m <= 256) sort_list<4>(l, g, b, m, lane);
    else if (m <= 512) sort_list<8>(l, g, b, m, lane);
    else sort_list<16>(l, g, b, m, lane);
  }
}

// Keys of more items, a workgroup each: a bitonic sort in LDS, or, past its size, the key's items
// picked from all of the group's in order (there are few such keys, whatever the input).
__global__ void __launch_bounds__(kHugeBlock) k_list_huge(Lists l) {
  __shared__ uint32_t v[kHugeLds];
  __shared__ int part[kHugeBlock / 64];
  const int n = l.n_longer[1];
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
    const int64_t key = l.huge[i], b = l.starts[key];
    const int64_t m = l.starts[key + 1] - b;
    const int g = group_of(l.keys, key);
    const int64_t at = b - l.starts[l.keys[g]];
    if (m <= kHugeLds) {
      int size = 2 * kWaveMax;
      while (size < m) size <<= 1;
      for (int k = threadIdx.x; k < size; k += kHugeBlock) v[k] = k < m ? l.unsorted[b + k] : ~0u;
      for (int k = 2; k <= size; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
          __syncthreads();
          for (int t = threadIdx.x; t < size / 2; t += kHugeBlock) {
            const int lo = 2 * t - (t & (j - 1)), hi = lo + j;
            const uint32_t a = v[lo], c = v[hi];
            if ((a > c) == ((lo & k) == 0)) {
              v[lo] = c;
              v[hi] = a;
            }
          }
        }
      __syncthreads();
      for (int k = threadIdx.x; k < m; k += kHugeBlock) put(l, g, at + k, v[k]);
    } else {
      const int64_t all = l.items[g + 1] - l.items[g];
      int64_t done = 0;
      for (int64_t x0 = 0; x0 < all; x0 += kHugeBlock * kHugeStream) {
        const int64_t x = x0 + (int64_t)threadIdx.x * kHugeStream;
        unsigned mine = 0;
        for (int u = 0; u < kHugeStream; ++u)
          if (x + u < all && key_of(l, g, x + u) == key) mine |= 1u << u;
        int total;
        int64_t to = at + done + block_exclusive_scan<int, kHugeBlock>(__popc(mine), part, &total);
        for (int u = 0; u < kHugeStream; ++u)
          if (mine >> u & 1) put(l, g, to++, x + u);
        done += total;
      }
    }
    __syncthreads();  // v is filled again
  }
}

// The first pair of every target (pairs are in target order), and the targets whose pairs are not
// all in one block of pairs (in no order: each is worked on by itself).
__global__ void __launch_bounds__(kBlock) k_targets(const int64_t* __restrict__ tt, int64_t n_pairs, int64_t n_tgt,
                                                    int64_t* __restrict__ offsets, int64_t* __restrict__ rest,
                                                    unsigned long long* n_rest) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t > n_tgt) return;
  auto first = [&](int64_t target) {
    int64_t lo = 0, hi = n_pairs;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (tt[mid] < target) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  const int64_t b = first(t);
  offsets[t] = b;
  if (t == n_tgt) return;
  const int64_t e = first(t + 1);
  const bool left = !whole_in_block(b, e);
  const uint64_t mask = __ballot(left);
  if (!mask) return;
  const int lane = lane_id(), lead = __ffsll((unsigned long long)mask) - 1;
  unsigned long long at = 0;
  if (lane == lead) at = atomicAdd(n_rest, (unsigned long long)__popcll(mask));
  at = __shfl(at, lead);
  if (left) rest[at + __popcll(mask & ((1ull << lane) - 1))] = t;
}

// Workspace: counts and the two counters (cleared together), starts, unsorted, rank, longer, huge, scan.
struct ListWs {
  int64_t keys, items;
  size_t counts, starts, unsorted, rank, longer, huge, scan, total;
  int64_t clear;  // int64 words from `counts`
};

ListWs carve_lists(const ct_regrid_topology* t) {
  ListWs w{};
  w.keys = t->n_src + t->n_tgt_vertices + t->n_src_vertices;
  w.items = t->n_pairs + t->n_tgt * t->n_max_t + t->n_src * t->n_max_s;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at += (bytes + 255) & ~size_t(255);
    return p;
  };
  w.clear = w.keys + 1;
  w.counts = take(sizeof(int64_t) * w.clear);
  w.starts = take(sizeof(int64_t) * (w.keys + 1));
  w.unsorted = take(sizeof(uint32_t) * w.items);
  w.rank = take(sizeof(uint32_t) * w.items);
  w.longer = take(sizeof(int32_t) * (w.items / kCompare + 1));
  w.huge = take(sizeof(int32_t) * (w.items / kWaveMax + 1));
  w.scan = take(ct_scan_workspace_bytes(w.keys));
  w.total = at;
  return w;
}

}  // namespace
}  // namespace ct

using namespace ct;

extern "C" {

size_t ct_regrid_lists_workspace_bytes(const ct_regrid_topology* topo) { return topo ? carve_lists(topo).total : 0; }

int ct_regrid_lists(const ct_regrid_topology* topo, void* workspace, size_t workspace_bytes, int64_t* tgt_offsets,
                    int64_t* src_offsets, int64_t* perm_by_src, int64_t* src_tgt, int64_t* tgt_vertex_offsets,
                    int64_t* tgt_vertex_corners, int64_t* src_vertex_offsets, int64_t* src_vertex_corners,
                    int64_t* rest_targets, int64_t* info, void* stream) {
  CT_REQUIRE(topo && topo->n_pairs >= 0 && topo->n_tgt >= 0 && topo->n_src >= 1 && topo->n_tgt_vertices >= 0 &&
                 topo->n_src_vertices >= 1 && topo->n_max_t >= 1 && topo->n_max_s >= 1,
             "bad sizes");
  CT_REQUIRE(topo->src_faces && (topo->n_tgt == 0 || (topo->tgt_faces && rest_targets)) &&
                 (topo->n_pairs == 0 || (topo->tt && topo->ss && perm_by_src && src_tgt)),
             "null arrays");
  CT_REQUIRE(tgt_offsets && src_offsets && tgt_vertex_offsets && src_vertex_offsets && src_vertex_corners && info &&
                 (topo->n_tgt == 0 || tgt_vertex_corners),
             "null outputs");
  const ListWs w = carve_lists(topo);
  // an item's number within its group, its rank and a list's length are 32-bit words
  CT_REQUIRE(topo->n_pairs < ((int64_t)1 << 31) && topo->n_tgt * topo->n_max_t < ((int64_t)1 << 31) &&
                 topo->n_src * topo->n_max_s < ((int64_t)1 << 31) && w.keys < (int64_t)kNone,
             "fewer than 2^31 pairs, target corners and source corners each");
  if (workspace_bytes < w.total) {
    set_error("list workspace too small: %zu < %zu", workspace_bytes, w.total);
    return CT_ERR_WORKSPACE;
  }
  hipStream_t st = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
  Lists l{};
  l.ss = topo->ss;
  l.tt = topo->tt;
  l.faces[0] = topo->tgt_faces;
  l.faces[1] = topo->src_faces;
  const int64_t nk[kGroups] = {topo->n_src, topo->n_tgt_vertices, topo->n_src_vertices};
  const int64_t ni[kGroups] = {topo->n_pairs, topo->n_tgt * topo->n_max_t, topo->n_src * topo->n_max_s};
  int64_t* const offsets[kGroups] = {src_offsets, tgt_vertex_offsets, src_vertex_offsets};
  int64_t* const list[kGroups] = {perm_by_src, tgt_vertex_corners, src_vertex_corners};
  for (int g = 0; g < kGroups; ++g) {
    l.keys[g + 1] = l.keys[g] + nk[g];
    l.items[g + 1] = l.items[g] + ni[g];
    l.offsets[g] = offsets[g];
    l.list[g] = list[g];
  }
  l.src_tgt = src_tgt;
  l.counts = reinterpret_cast<int64_t*>(ws + w.counts);
  l.n_longer = reinterpret_cast<int32_t*>(l.counts + w.keys);
  l.starts = reinterpret_cast<int64_t*>(ws + w.starts);
  l.unsorted = reinterpret_cast<uint32_t*>(ws + w.unsorted);
  l.rank = reinterpret_cast<uint32_t*>(ws + w.rank);
  l.longer = reinterpret_cast<uint32_t*>(ws + w.longer);
  l.huge = reinterpret_cast<uint32_t*>(ws + w.huge);
  int rc = fill<int64_t>(l.counts, w.clear, 0, st);
  if (!rc) rc = fill<int64_t>(info, 3, 0, st);
  // a group without keys writes no offset by k_list_rank
  if (!rc && topo->n_tgt_vertices == 0) rc = fill<int64_t>(tgt_vertex_offsets, 1, 0, st);
  if (rc) return rc;
  k_targets<<<grid_for(topo->n_tgt + 1), kBlock, 0, st>>>(topo->tt, topo->n_pairs, topo->n_tgt, tgt_offsets, rest_targets,
                                                        reinterpret_cast<unsigned long long*>(info));
  auto grid = [](int64_t all, int64_t x0) { return grid_for(std::min(all - x0, kItemsPerLaunch)); };
  for (int64_t x0 = 0; x0 < w.items; x0 += kItemsPerLaunch)
    k_list_count<<<grid(w.items, x0), kBlock, 0, st>>>(l, x0);
  CT_LAUNCH_CHECK();
  rc = exclusive_scan(l.counts, w.keys, l.starts, ws + w.scan, ct_scan_workspace_bytes(w.keys), st);
  if (rc) return rc;
  for (int64_t x0 = 0; x0 < w.items; x0 += kItemsPerLaunch)
    k_list_place<<<grid(w.items, x0), kBlock, 0, st>>>(l, x0);
  for (int64_t x0 = 0; x0 < std::max(w.items, w.keys); x0 += kItemsPerLaunch)
    k_list_rank<<<grid(std::max(w.items, w.keys), x0), kBlock, 0, st>>>(l, x0, info);
  k_list_longer<<<1024, kBlock, 0, st>>>(l);
  k_list_huge<<<256, kHugeBlock, 0, st>>>(l);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

}  // extern "C"
