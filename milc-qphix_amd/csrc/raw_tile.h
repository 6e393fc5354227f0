// raw_tile.h -- 64 sites of a raw link array (72 reals a site) in LDS, loaded and
// stored as whole lines by a block of 256.
#pragma once
#include "device.h"

namespace qphix {

// Reals from one site to the next in LDS: two more than 72, so that lanes at
// consecutive sites reading one element spread over the banks (16-byte aligned).
constexpr int RAW_TILE_STRIDE = 74;
constexpr int RAW_TILE_REALS = 64 * RAW_TILE_STRIDE;

// Every raw transfer holds whole tiles: the sites of a parity are a multiple of
// 128, a chunk's a multiple of 64 (hostio.hip).
template <typename T> __device__ __forceinline__ void raw_tile_in(T *tile, const T *raw) {
  using T2 = typename std::conditional<sizeof(T) == 8, double2, float2>::type;
  const T2 *s = reinterpret_cast<const T2 *>(raw);
  T2 *d = reinterpret_cast<T2 *>(tile);
#pragma unroll
  for (int k = 0; k < 9; ++k) {  // 64 sites x 36 complex numbers
    const int e = k * 256 + (int)threadIdx.x;
    d[(e / 36) * (RAW_TILE_STRIDE / 2) + e % 36] = s[e];
  }
  __syncthreads();
}

template <typename T> __device__ __forceinline__ void raw_tile_out(T *raw, const T *tile) {
  using T2 = typename std::conditional<sizeof(T) == 8, double2, float2>::type;
  __syncthreads();
  const T2 *s = reinterpret_cast<const T2 *>(tile);
  T2 *d = reinterpret_cast<T2 *>(raw);
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int e = k * 256 + (int)threadIdx.x;
    d[e] = s[(e / 36) * (RAW_TILE_STRIDE / 2) + e % 36];
  }
}

} // namespace qphix
