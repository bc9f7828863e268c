// ct_primitives.h -- wavefront / workgroup building blocks (64-lane wavefronts, 256-lane
// workgroups).  No hipMemsetAsync anywhere: buffers are cleared by kernels so that every
// entry point stays safe to capture in a HIP graph.
#pragma once

#include "ct_internal.h"

namespace ct {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// Exclusive scan over a BLOCK-lane workgroup (BLOCK a multiple of 64, at most 1024).  lds
// must hold BLOCK/64 elements.  Every lane must call it (it contains barriers).  *total
// receives the workgroup sum.
template <typename T, int BLOCK = kBlock>
__device__ __forceinline__ T block_exclusive_scan(T v, T* lds, T* total) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  T x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) lds[w] = x;
  __syncthreads();
  T before = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < BLOCK / 64; ++k) {
    const T s = lds[k];
    if (k < w) before += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return before + x - v;
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

template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t n, T value) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

template <typename T>
inline int fill(T* p, int64_t n, T value, hipStream_t st) {
  if (n <= 0) return CT_OK;
  k_fill<T><<<grid_for(n), kBlock, 0, st>>>(p, n, value);
  CT_LAUNCH_CHECK();
  return CT_OK;
}

// celltree_base.py:20-48 on n boxes: distances (n, 3) when not null, and 5 keys reduced from 0
// (~min x, max x, ~min y, max y, max diagonal as order-preserving keys; ct_geometry.hip).
int bbox_stat_keys(const double* bb, int64_t n, double* distances, unsigned long long* keys, hipStream_t st);

int exclusive_scan(const int64_t* in, int64_t n, int64_t* out, void* ws, size_t ws_bytes,
                   hipStream_t st);

}  // namespace ct
