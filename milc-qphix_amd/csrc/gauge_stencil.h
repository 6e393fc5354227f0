// gauge_stencil.h -- site order and neighbour arithmetic of the gauge-field
// kernels (staple products of the gauge force, smearing of the fermion links).
#pragma once
#include "common.h"

namespace qphix {

struct GqGeo {
  int L[4];
  int nxh, vh;
  int stride[4];  // lexicographic strides 1, L0, L0 L1, L0 L1 L2
  int zreg;       // 1: each XCD's slab of site blocks is a z-region (gq_site)
};

// Site of logical index Lg: itself, or with zreg the XCD x = Lg / (vh / 8)
// takes the z-planes [x nz / 8, (x + 1) nz / 8) t-slice by t-slice, so the 8
// XCDs advance through t together and the +-1 neighbourhood they read is a
// few planes of each region instead of whole t-slices.
__device__ __forceinline__ int gq_site(const GqGeo &g, int Lg) {
  if (!g.zreg) return Lg;
  const int nxy = g.nxh * g.L[1], nzl = g.L[2] / 8;
  const int per = nxy * nzl * g.L[3], slice = nxy * nzl;
  const int x = Lg / per;
  int r = Lg - x * per;
  const int t = r / slice;
  r -= t * slice;
  const int z = x * nzl + r / nxy;
  return (r % nxy) + nxy * (z + g.L[2] * t);
}

// Coordinates of half-site i of parity cb.
__device__ __forceinline__ void q_coords(const GqGeo &g, int i, int cb, int c[4]) {
  const int xh = i % g.nxh;
  int r = i / g.nxh;
  c[1] = r % g.L[1];
  r /= g.L[1];
  c[2] = r % g.L[2];
  c[3] = r / g.L[2];
  c[0] = 2 * xh + ((c[1] + c[2] + c[3] + cb) & 1);
}

// Coordinate of direction d (uniform) without indexing a per-lane array.
__device__ __forceinline__ int q_coord(const int c[4], int d) {
  return d == 0 ? c[0] : d == 1 ? c[1] : d == 2 ? c[2] : c[3];
}

// Lexicographic index r moved by s (+-1) along d (uniform), coordinate cd
// along d before the move; wraps periodically.
__device__ __forceinline__ int q_move(const GqGeo &g, int r, int cd, int d, int s) {
  const int L = g.L[d], st = g.stride[d];
  const int v = cd + s;
  r += s * st;
  if (v < 0) r += L * st;
  else if (v >= L) r -= L * st;
  return r;
}

// The three directions other than mu, in increasing order; rank of d among
// the directions other than m.
__device__ __forceinline__ int q_other(int mu, int k) { return k < mu ? k : k + 1; }
__device__ __forceinline__ int q_rank(int m, int d) { return d < m ? d : d - 1; }

// Block -> slot: each XCD (blocks are dispatched round-robin over 8 XCDs)
// sweeps one contiguous slab of slots.
__device__ __forceinline__ int gq_slot() {
  const int nb = gridDim.x, b = blockIdx.x;
  return nb % 8 == 0 ? (b % 8) * (nb / 8) + b / 8 : b;
}

// This lattice in site order (zreg = 0).
inline GqGeo gq_geo() {
  const Geometry &gg = ctx().g;
  GqGeo g{};
  g.L[0] = gg.nx;
  g.L[1] = gg.ny;
  g.L[2] = gg.nz;
  g.L[3] = gg.nt;
  g.nxh = gg.nxh;
  g.vh = gg.vh;
  g.stride[0] = 1;
  g.stride[1] = gg.nx;
  g.stride[2] = gg.nx * gg.ny;
  g.stride[3] = gg.nx * gg.ny * gg.nz;
  return g;
}

} // namespace qphix
