// A step's rows cut into tiles of equal size that never cross a request: which tile a block works on.
#pragma once

#include "common.h"

namespace tk {

struct RequestTile {
  int req, index;      // the request, and the tile's number within it
};

// Tiles of `size` rows of a request; none where it brings fewer than `least` rows (another kernel's work).
__device__ __forceinline__ int request_tiles(const int* __restrict__ q_start, int req, int size, int least) {
  const int rows = q_start[req + 1] - q_start[req];
  return rows >= least ? (rows + size - 1) / size : 0;
}

// The tiles of the requests before `req`.  All lanes of a wave must call, each wave counts for itself.
__device__ __forceinline__ int tiles_before(const int* __restrict__ q_start, int req, int size, int least) {
  int count = 0;
  for (int r = threadIdx.x & (kWave - 1); r < req; r += kWave) count += request_tiles(q_start, r, size, least);
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) count += __shfl_xor(count, m, kWave);
  return __builtin_amdgcn_readfirstlane(count);
}

// Tile number `at` of the step, the requests' tiles of `size` rows counted in their order; false past the last one.
// Every wave counts for itself (all its lanes must call): 64 requests a turn, a prefix sum over the lanes.
__device__ __forceinline__ bool find_request_tile(const int* __restrict__ q_start, int requests, int size, int at, RequestTile& t,
                                                  int least = 1) {
  const int lane = threadIdx.x & (kWave - 1);
  int before = 0;
  for (int base = 0; base < requests; base += kWave) {
    const int r = base + lane;
    const int count = r < requests ? request_tiles(q_start, r, size, least) : 0;
    int upto = count;
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
      const int other = __shfl_up(upto, m, kWave);
      if (lane >= m) upto += other;
    }
    const int total = __shfl(upto, kWave - 1, kWave);
    if (at < before + total) {
      const unsigned long long mine = __ballot(at >= before + upto - count && at < before + upto);
      const int owner = __ffsll(mine) - 1;
      t.req = __builtin_amdgcn_readfirstlane(base + owner);
      t.index = __builtin_amdgcn_readfirstlane(at - __shfl(before + upto - count, owner, kWave));
      return true;
    }
    before += total;
  }
  return false;
}

}  // namespace tk
