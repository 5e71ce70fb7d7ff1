// scan.hpp -- one-block exclusive scan of the neighbour list's cell counts:
// start[i] = base + sum_{j<i} count[j], start[n] = base + total; the counts
// are cleared for the next use.  They may have been written by other blocks'
// atomics, so they are read past the caches.  Call with all threads of a
// block (<= 1024 threads, multiple of 64).  True in a thread that met a count
// above `most`.
#pragma once
#include <hip/hip_runtime.h>

namespace mmamd {

constexpr int SCAN_PER = 8;   // consecutive counts per thread and round

__device__ inline bool block_scan_clear(int *count, int *start, int n, int base, int most) {
  __shared__ int wsum[16];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int carry = base;
  bool above = false;
  for (int b = 0; b < n; b += SCAN_PER * blockDim.x) {
    const int c = b + SCAN_PER * threadIdx.x;
    int v[SCAN_PER], sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER; k++)
      v[k] = c + k < n ? __hip_atomic_load(count + c + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER; k++) {
      sum += v[k];
      above |= v[k] > most;
    }
    int x = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wid] = x;
    __syncthreads();
    int at = carry + x - sum;
    for (int w = 0; w < nw; w++) {
      if (w < wid) at += wsum[w];
      carry += wsum[w];
    }
#pragma unroll
    for (int k = 0; k < SCAN_PER; k++) {
      if (c + k < n) {
        start[c + k] = at;
        count[c + k] = 0;
      }
      at += v[k];
    }
    __syncthreads();   // the next round writes wsum
  }
  if (threadIdx.x == 0) start[n] = carry;
  return above;
}

}  // namespace mmamd
