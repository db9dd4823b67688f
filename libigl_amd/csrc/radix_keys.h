// radix_keys.h -- keys of a batch of queries, counted as they are made
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace gwn {

constexpr int RS_THREADS = 256;
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = RS_THREADS * RS_ITEMS;

// keys[i] = key(i) for i < n, and each sort tile's counts of the keys' lowest
// eight bits (what k_rs_tile_hist counts for the first pass), so that the sort
// need not read the keys for them (5.3 us and a launch per 1M), nor write and
// read values that are the keys' positions.  One block per tile, of 1,024
// threads: with the sort's 256 a batch of 1M fills less of the chip (2D keys
// 8.2 us, now 7.1; 3D Hilbert keys 13.0, now 12.6, bound by their ~300
// instructions).  1M queries, whole calls: curve 165 -> 160 us, antipodal 296
// -> 282.  vals[0] is written for the batch of one, which the sort leaves as
// it is.
constexpr int RS_KEY_THREADS = 1024;
template <typename KeyFn>
__global__ __launch_bounds__(RS_KEY_THREADS) void k_rs_keys(KeyFn key, int64_t n, uint32_t* __restrict__ keys,
                                                            uint32_t* __restrict__ vals,
                                                            uint32_t* __restrict__ counts, int64_t nt) {
  __shared__ uint32_t h[256];
  if (threadIdx.x < 256) h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * RS_TILE;
#pragma unroll
  for (int r = 0; r < RS_TILE / RS_KEY_THREADS; ++r) {
    const int64_t i = base + r * RS_KEY_THREADS + threadIdx.x;
    if (i < n) {
      const uint32_t k = key(i);
      keys[i] = k;
      atomicAdd(&h[k & 0xFFu], 1u);
    }
  }
  if (n == 1 && threadIdx.x == 0) vals[0] = 0;
  __syncthreads();
  if (threadIdx.x < 256) counts[(int64_t)threadIdx.x * nt + blockIdx.x] = h[threadIdx.x];
}

}  // namespace gwn
