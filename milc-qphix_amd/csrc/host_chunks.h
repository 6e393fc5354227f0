// host_chunks.h -- how a transfer of raw host arrays is cut into chunks of sites
// (hostio.hip).  Plain C++, without the device.
#pragma once
#include <algorithm>
#include <cstddef>

namespace qphix {

constexpr size_t HOST_CHUNK = (size_t)8 << 20;  // bytes of one pinned buffer: the most of a chunk
constexpr size_t HOST_CHUNK_MIN = (size_t)1 << 20;
constexpr int HOST_BUFS = 4;  // buffers of the ring
// Up to here the conversion kernels read and write the pinned buffers
// themselves: one launch a chunk and no staging in device memory.
constexpr size_t HOST_DIRECT = (size_t)4 << 20;

// Bytes that a chunk aims at: a quarter of a small transfer, so that its chunks overlap.
inline size_t host_chunk_bytes(size_t per_site, size_t half, int halves) {
  return std::min(HOST_CHUNK, std::max(HOST_CHUNK_MIN, per_site * half * halves / 4));
}

struct HostPlan {
  size_t per_site = 0, half = 0, chunk = 0;  // bytes of a site over all arrays; sites of a half, of a chunk
  size_t per_half = 0, chunks = 0;           // chunks of a half, of the transfer
  bool direct = false;                       // the kernels use the pinned buffers themselves
  int nbuf = 1;
  size_t first(size_t c) const { return c / per_half * half + c % per_half * chunk; }
  size_t count(size_t c) const { return std::min(chunk, half - c % per_half * chunk); }
};

inline HostPlan host_plan(size_t per_site, size_t half, int halves) {
  HostPlan p;
  p.per_site = per_site;
  p.half = half;
  p.chunk = std::min(half, std::max<size_t>(64, host_chunk_bytes(per_site, half, halves) / per_site / 64 * 64));
  p.per_half = (half + p.chunk - 1) / p.chunk;
  p.chunks = p.per_half * halves;
  p.direct = per_site * half * halves <= HOST_DIRECT;
  p.nbuf = (int)std::min<size_t>(HOST_BUFS, p.chunks);
  return p;
}

// Device staging of a transfer.  It also holds a transfer of fewer bytes a site
// over the same sites (some of the arrays alone): whole buffers of the size that
// a chunk aims at, not of the chunk, whose rounding to 64 sites differs.
inline size_t host_stage_bytes(size_t per_site, size_t half, int halves) {
  if (host_plan(per_site, half, halves).chunk == half) return per_site * half * halves;
  return HOST_BUFS * std::max(host_chunk_bytes(per_site, half, halves), 64 * per_site);
}

} // namespace qphix
