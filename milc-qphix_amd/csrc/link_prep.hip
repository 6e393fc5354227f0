// link_prep.hip -- asqtad / HISQ fermion links from the thin gauge field, on
// the device.
//
// In the reference the smeared links arrive from MILC (asqtad_create_L_from_raw,
// qphix_d3.cpp:970-1085) with the staggered phases already folded in; its own
// rephase and long-link kernels are disabled (ks_dslash_complete_specialization
// .cpp:238-275, `#if 0`).  Here they are built from a GaugeField (SU(3) links,
// no phases) on the GPU:
//
//   fat_mu(x) = eta_mu(x) b_mu(x) [ c1 U_mu(x) + sum over staple paths ],
//   lng_mu(x) = eta_mu(x) b3_mu(x) cN U_mu(x) U_mu(x+mu) U_mu(x+2mu),
//
// with the paths of Orginos, Toussaint & Sugar (Phys. Rev. D 60 (1999) 054503)
// and Lepage (Phys. Rev. D 59 (1999) 074502): 6 three-link staples (weight c3
// each), 24 five-link and 48 seven-link staples (c5, c7 per ordered path) and
// 6 five-link Lepage paths (cL), written with the physical (unphased) signs:
// fat7 = (1/8, 1/16, 1/64, 1/384), asqtad adds cL = -1/16, cN = -1/24 and
// c1 = 5/8.  The staples are nested: with the staple map
//   S_{d,s}(M)(y) = U_d(y) M(y+d) U_d(y+mu)^dag          (s = +1)
//                 = U_d(y-d)^dag M(y-d) U_d(y-d+mu)       (s = -1),
//   fat = c1 U + sum_{d,s} S_{d,s}( c3 U + cL S_{d,s}(U)
//                  + sum_{e,s'} S_{e,s'}( c5 U + c7 sum_{f,s''} S_{f,s''}(U) ) ),
// d, e, f distinct directions other than mu.  An inner staple sum is needed by
// every link around it, so each level of the nest is formed once per link and
// stored (smear_level): 48 SU(3) products per link, 60 with Lepage paths,
// against 168 when every link forms its own nest.
// eta_mu(x) is MILC's staggered phase (C11: (-1)^t, (-1)^(t+x), (-1)^(t+x+y),
// 1); b_mu = -1 on t-links whose path crosses the last time slice when the
// time boundary is antiperiodic (the phases and the boundary commute with the
// smearing: every path from x to x+mu carries the same signs).  Back links are
// MILC's double store, slot 2mu at x = -fwd_mu(x - hop mu)^dag.
//
// HISQ (Follana et al., Phys. Rev. D 75 (2007) 054502): W = P_U(3)(fat7(U)),
// the unitary projection V (V^dag V)^(-1/2) (here the polar factor, by the
// scaled Newton iteration X <- (z X + (z X)^(-dag)) / 2, z = |det X|^(-1/3)
// (Higham, SIAM J. Sci. Stat. Comput. 7 (1986) 1160)); then the fat links are
// the asqtad-like smearing of W with c1 = 1, c3 = 1/16, c5 = 1/64, c7 = 1/384,
// cL = -1/8, and the Naik links -1/24 (1 + eps_N) W W W.
//
// The phased fat/long links and back links go straight into the tile-major
// pairs of a link handle (k_links_pack); the Naik storage (12 or 18 reals) is
// decided by the test that links handed over by MILC undergo (fields.hip).
#include "blas.h"
#include "gauge_stencil.h"
#include "handles.h"
#include "qphix_mi355x.h"

#include <chrono>

namespace qphix {

struct CM3 {
  double re[9], im[9];
};

// r = a^(dag if DA) * b^(dag if DB), or with ACC r += c times that.  An element's
// product is summed from zero and then added in one step: summed on top of r,
// every partial product would be rounded at the size of r (fat links 1.3e-16 ->
// 2.8e-16 rms against extended precision).
template <bool DA, bool DB, bool ACC>
__device__ __forceinline__ void cm_product(const CM3 &a, const CM3 &b, double c, CM3 &r) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double sr = 0, si = 0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int ia = DA ? 3 * k + i : 3 * i + k, ib = DB ? 3 * j + k : 3 * k + j;
        const double ar = a.re[ia], ai = DA ? -a.im[ia] : a.im[ia];
        const double br = b.re[ib], bi = DB ? -b.im[ib] : b.im[ib];
        sr = fma(ar, br, sr);
        sr = fma(-ai, bi, sr);
        si = fma(ar, bi, si);
        si = fma(ai, br, si);
      }
      r.re[3 * i + j] = ACC ? fma(c, sr, r.re[3 * i + j]) : sr;
      r.im[3 * i + j] = ACC ? fma(c, si, r.im[3 * i + j]) : si;
    }
}

template <bool DA, bool DB> __device__ __forceinline__ void cm_mul(const CM3 &a, const CM3 &b, CM3 &r) {
  cm_product<DA, DB, false>(a, b, 1.0, r);
}

template <bool DA, bool DB> __device__ __forceinline__ void cm_madd(double c, const CM3 &a, const CM3 &b, CM3 &r) {
  cm_product<DA, DB, true>(a, b, c, r);
}

__device__ __forceinline__ void cm_zero(CM3 &a) {
#pragma unroll
  for (int e = 0; e < 9; ++e) a.re[e] = a.im[e] = 0;
}

__device__ __forceinline__ void cm_add(const CM3 &a, CM3 &r) {
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    r.re[e] += a.re[e];
    r.im[e] += a.im[e];
  }
}

__device__ __forceinline__ void cm_scale(double c, CM3 &a) {
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    a.re[e] *= c;
    a.im[e] *= c;
  }
}

// Matrix m of half-site i of one parity of a field in the gauge layout:
// element e is the complex number (m*9 + e)*vh + i.
template <typename T> __device__ __forceinline__ void cm_load(const T *base, int m, int vh, int i, CM3 &a) {
  using T2 = typename std::conditional<sizeof(T) == 8, double2, float2>::type;
  const T2 *b = reinterpret_cast<const T2 *>(base) + (size_t)(m * 9) * (size_t)vh;
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    const T2 v = b[(size_t)e * (size_t)vh + i];
    a.re[e] = (double)v.x;
    a.im[e] = (double)v.y;
  }
}

// Streaming: what a pass writes is read by the next one only (24^4, against
// cached stores: the three passes 91 / 191 / 120 -> 84 / 174 / 109 us).
__device__ __forceinline__ void cm_store(double *base, int m, int vh, int i, const CM3 &a) {
  nd2 *b = reinterpret_cast<nd2 *>(base) + (size_t)(m * 9) * (size_t)vh;
#pragma unroll
  for (int e = 0; e < 9; ++e) __builtin_nontemporal_store(nd2{a.re[e], a.im[e]}, b + (size_t)e * (size_t)vh + i);
}

struct SmearCoef {
  double c1, c3, c5, c7, cl, cn;
};
// HISQ's second level (Follana et al. 2007): one link 1/8 + 2 * 3/8 + 1/8,
// staples as fat7, Lepage twice the asqtad value, Naik -(1 + eps)/24.
static SmearCoef hisq_level2(double naik_eps) {
  return SmearCoef{1.0, 1.0 / 16, 1.0 / 64, 1.0 / 384, -1.0 / 8, -(1.0 + naik_eps) / 24.0};
}

// ---------------------------------------------------------------------------
// One smearing level in three passes over the lattice, for the link directions
// mu0 .. mu0 + nmu - 1 together.  Slots of M and N: mu - mu0 first.
//   inner: M_{mu,f} = c5 U_mu + c7 sum_s S_{f,s}(U_mu)              3 per mu
//   mid:   N_{mu,d,s} = c3 U_mu + sum_{e,s'} S_{e,s'}(M_{mu,f}) [+ cL S_{d,s}(U_mu)]
//          (f the direction that is none of mu, d, e)   6 per mu, 3 without Lepage
//   outer: fat_mu = c1 U_mu + sum_{d,s} S_{d,s}(N_{mu,d,s}); the Naik links
// A work-item forms one matrix of one site (lanes run over consecutive sites,
// so every element is one contiguous wavefront access); the blocks of a site
// block's directions and parities are neighbours in their XCD's slab, so they
// share its links in L2.  A pass is bound by memory: per mu and site it moves
// 144 B x (4 thin links + 3) in the first pass, (4 + 3 + 6) in the second and
// (4 + 6 + 1 + 1) in the third, for 48 or 60 products per link.
// ---------------------------------------------------------------------------
struct SmearArgs {
  const void *u[2];  // thin links, parity 0 / 1 (gauge layout)
  double *m[2], *n[2];
  double *fat[2], *naik[2];  // naik null: not formed
  GqGeo g;
  SmearCoef k;
  int mu0, nmu;
  int lep;   // N has a slot for each sign (Lepage paths)
  int five;  // five- or seven-link staples present
};

// A site: half-site i of parity cb, its lexicographic index and coordinates,
// the thin links of its own and the other parity, and its neighbour x + mu.
template <typename T> struct SmearSite {
  const T *us, *uo;
  int i, r, mu, imu, rmu;
  int c[4];
};

template <typename T>
__device__ __forceinline__ void smear_site(const SmearArgs &a, int i, int cb, int mu, SmearSite<T> &x) {
  x.us = static_cast<const T *>(a.u[cb]);
  x.uo = static_cast<const T *>(a.u[1 - cb]);
  x.i = i;
  x.mu = mu;
  q_coords(a.g, i, cb, x.c);
  x.r = x.c[0] + a.g.L[0] * (x.c[1] + a.g.L[1] * (x.c[2] + a.g.L[2] * x.c[3]));
  x.rmu = q_move(a.g, x.r, q_coord(x.c, mu), mu, 1);
  x.imu = x.rmu >> 1;
}

// acc += c S_{d,+}(M)(x), M (matrix slot of the other parity's field mo) at x + d
template <typename T, typename TM>
__device__ __forceinline__ void staple_up(const GqGeo &g, const SmearSite<T> &x, int d, const TM *mo, int slot,
                                          double c, CM3 &acc) {
  CM3 A, M, t;
  cm_load(mo, slot, g.vh, q_move(g, x.r, q_coord(x.c, d), d, 1) >> 1, M);
  cm_load(x.us, d, g.vh, x.i, A);
  cm_mul<false, false>(A, M, t);
  cm_load(x.uo, d, g.vh, x.imu, A);
  cm_madd<false, true>(c, t, A, acc);
}

// acc += c S_{d,-}(M)(x), M at x - d
template <typename T, typename TM>
__device__ __forceinline__ void staple_down(const GqGeo &g, const SmearSite<T> &x, int d, const TM *mo, int slot,
                                            double c, CM3 &acc) {
  CM3 A, M, t;
  const int cd = q_coord(x.c, d);
  const int im = q_move(g, x.r, cd, d, -1) >> 1;
  cm_load(mo, slot, g.vh, im, M);
  cm_load(x.uo, d, g.vh, im, A);
  cm_mul<true, false>(A, M, t);
  cm_load(x.us, d, g.vh, q_move(g, x.rmu, cd, d, -1) >> 1, A);  // d is not mu: the coordinate is x's
  cm_madd<false, false>(c, t, A, acc);
}

// Block -> (site block, variant of nv), as gq_slot; false past the last site.
__device__ __forceinline__ bool smear_slot(const GqGeo &g, int nv, int &i, int &v) {
  const int slot = gq_slot();
  v = slot % nv;
  const int il = (slot / nv) * 256 + (int)threadIdx.x;
  if (il >= g.vh) return false;
  i = gq_site(g, il);
  return true;
}

template <typename T> __global__ void __launch_bounds__(256) k_smear_inner(const SmearArgs a) {
  int i, v;
  if (!smear_slot(a.g, 6 * a.nmu, i, v)) return;
  const int cb = v & 1, q = v >> 1, ml = q / 3, mu = a.mu0 + ml, fr = q % 3, f = q_other(mu, fr);
  SmearSite<T> x;
  smear_site<T>(a, i, cb, mu, x);
  CM3 acc;
  cm_load(x.us, mu, a.g.vh, i, acc);
  cm_scale(a.k.c5, acc);
  if (a.k.c7 != 0) {
    staple_up(a.g, x, f, x.uo, mu, a.k.c7, acc);
    staple_down(a.g, x, f, x.uo, mu, a.k.c7, acc);
  }
  cm_store(a.m[cb], 3 * ml + fr, a.g.vh, i, acc);
}

template <typename T> __global__ void __launch_bounds__(256) k_smear_mid(const SmearArgs a) {
  int i, v;
  if (!smear_slot(a.g, 6 * a.nmu, i, v)) return;
  const int cb = v & 1, q = v >> 1, ml = q / 3, mu = a.mu0 + ml, dr = q % 3, d = q_other(mu, dr);
  SmearSite<T> x;
  smear_site<T>(a, i, cb, mu, x);
  CM3 acc, n;
  if (!a.lep) {
    cm_load(x.us, mu, a.g.vh, i, acc);
    cm_scale(a.k.c3, acc);
  } else {
    cm_zero(acc);
  }
  if (a.five) {
#pragma unroll 1
    for (int j = 1; j < 3; ++j) {  // e, f: the other two directions, either way round
      const int er = (dr + j) % 3, fr = (dr + 3 - j) % 3;
      const int e = q_other(mu, er);
      staple_up(a.g, x, e, a.m[1 - cb], 3 * ml + fr, 1.0, acc);
      staple_down(a.g, x, e, a.m[1 - cb], 3 * ml + fr, 1.0, acc);
    }
  }
  if (!a.lep) {
    cm_store(a.n[cb], 3 * ml + dr, a.g.vh, i, acc);
    return;
  }
  // the three-link and Lepage terms, of opposite signs, before the rest
#pragma unroll
  for (int up = 1; up >= 0; --up) {
    cm_load(x.us, mu, a.g.vh, i, n);
    cm_scale(a.k.c3, n);
    if (up) staple_up(a.g, x, d, x.uo, mu, a.k.cl, n);
    else staple_down(a.g, x, d, x.uo, mu, a.k.cl, n);
    cm_add(acc, n);
    cm_store(a.n[cb], 2 * (3 * ml + dr) + 1 - up, a.g.vh, i, n);
  }
}

template <typename T> __global__ void __launch_bounds__(256) k_smear_outer(const SmearArgs a) {
  int i, v;
  if (!smear_slot(a.g, 2 * a.nmu, i, v)) return;
  const int cb = v & 1, ml = v >> 1, mu = a.mu0 + ml;
  SmearSite<T> x;
  smear_site<T>(a, i, cb, mu, x);
  CM3 acc;
  cm_load(x.us, mu, a.g.vh, i, acc);
  if (a.naik[0]) {  // cN U_mu(x) U_mu(x+mu) U_mu(x+2mu)
    const int c1 = q_coord(x.c, mu) + 1;
    CM3 b, p, nk;
    cm_load(x.uo, mu, a.g.vh, x.imu, b);
    cm_mul<false, false>(acc, b, p);
    cm_load(x.us, mu, a.g.vh, q_move(a.g, x.rmu, c1 >= a.g.L[mu] ? 0 : c1, mu, 1) >> 1, b);
    cm_mul<false, false>(p, b, nk);
    cm_scale(a.k.cn, nk);
    cm_store(a.naik[cb], mu, a.g.vh, i, nk);
  }
  cm_scale(a.k.c1, acc);
#pragma unroll 1
  for (int dr = 0; dr < 3; ++dr) {
    const int d = q_other(mu, dr), q = 3 * ml + dr;
    staple_up(a.g, x, d, a.n[1 - cb], a.lep ? 2 * q : q, 1.0, acc);
    staple_down(a.g, x, d, a.n[1 - cb], a.lep ? 2 * q + 1 : q, 1.0, acc);
  }
  cm_store(a.fat[cb], mu, a.g.vh, i, acc);
}

// 3x3 complex inverse by cofactors: r = a^-1.
__device__ __forceinline__ void cm_inv(const CM3 &a, CM3 &r) {
  // cofactor C_ij (complex); inverse = C^T / det
  double cr[9], ci[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      // a[i1][j1] a[i2][j2] - a[i1][j2] a[i2][j1]
      const double pr = a.re[3 * i1 + j1] * a.re[3 * i2 + j2] - a.im[3 * i1 + j1] * a.im[3 * i2 + j2];
      const double pi = a.re[3 * i1 + j1] * a.im[3 * i2 + j2] + a.im[3 * i1 + j1] * a.re[3 * i2 + j2];
      const double qr = a.re[3 * i1 + j2] * a.re[3 * i2 + j1] - a.im[3 * i1 + j2] * a.im[3 * i2 + j1];
      const double qi = a.re[3 * i1 + j2] * a.im[3 * i2 + j1] + a.im[3 * i1 + j2] * a.re[3 * i2 + j1];
      cr[3 * i + j] = pr - qr;
      ci[3 * i + j] = pi - qi;
    }
  double dr = 0, di = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    dr += a.re[j] * cr[j] - a.im[j] * ci[j];
    di += a.re[j] * ci[j] + a.im[j] * cr[j];
  }
  const double n = dr * dr + di * di;
  const double ir = dr / n, ii = -di / n;  // 1 / det
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double xr = cr[3 * j + i], xi = ci[3 * j + i];
      r.re[3 * i + j] = xr * ir - xi * ii;
      r.im[3 * i + j] = xr * ii + xi * ir;
    }
}

__device__ __forceinline__ double cm_absdet(const CM3 &a) {
  double dr = 0, di = 0;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int j1 = (j + 1) % 3, j2 = (j + 2) % 3;
    const double pr = a.re[3 + j1] * a.re[6 + j2] - a.im[3 + j1] * a.im[6 + j2];
    const double pi = a.re[3 + j1] * a.im[6 + j2] + a.im[3 + j1] * a.re[6 + j2];
    const double qr = a.re[3 + j2] * a.re[6 + j1] - a.im[3 + j2] * a.im[6 + j1];
    const double qi = a.re[3 + j2] * a.im[6 + j1] + a.im[3 + j2] * a.re[6 + j1];
    const double cr = pr - qr, ci = pi - qi;
    dr += a.re[j] * cr - a.im[j] * ci;
    di += a.re[j] * ci + a.im[j] * cr;
  }
  return sqrt(dr * dr + di * di);
}

// a / z from iz = 1 / z: the product and one correction by its remainder
// (Markstein, IBM J. Res. Dev. 34 (1990) 111), which rounds as a quotient does.
__device__ __forceinline__ double quotient(double a, double z, double iz) {
  const double q = a * iz;
  return fma(fma(-q, z, a), iz, q);
}

// Unitary polar factor of every link, in place (gauge layout, FP64): scaled
// Newton iterations until the update is below 1e-15 (at most 30).  One
// work-item per link, consecutive sites of a direction in consecutive lanes.  Its
// time is the FP64 arithmetic of four to six iterations; a cube root and one
// reciprocal an iteration, where it was pow and 18 quotients, took 24^4 from 177
// to about 95 us.  The elements are divided to a quotient's rounding all the same:
// scaled by the rounded reciprocal, W drifted off unitarity (HISQ Naik links of
// smooth fields 2.0e-16 rms from extended precision, against 1.6e-16 either way
// of dividing; 5 us of the 3.41 ms that rebuilding 24^4 HISQ links takes).
__global__ void __launch_bounds__(256) k_u3_project(double *v0, double *v1, int vh) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  const int mu = blockIdx.y & 3;
  double *v = (blockIdx.y >> 2) ? v1 : v0;
  CM3 X;
  cm_load(v, mu, vh, i, X);
  for (int it = 0; it < 30; ++it) {
    const double z = rcbrt(cm_absdet(X)), iz = 1.0 / z;
    CM3 Xi;
    cm_inv(X, Xi);
    double delta = 0;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        // (z X + (z X)^(-dag)) / 2; (X^-1)^dag element (r, c) = conj(Xi(c, r))
        const double yr = quotient(Xi.re[3 * c + r], z, iz), yi = quotient(Xi.im[3 * c + r], z, iz);
        const double nr = 0.5 * (z * X.re[3 * r + c] + yr);
        const double ni = 0.5 * (z * X.im[3 * r + c] - yi);
        delta = fmax(delta, fabs(nr - X.re[3 * r + c]) + fabs(ni - X.im[3 * r + c]));
        X.re[3 * r + c] = nr;
        X.im[3 * r + c] = ni;
      }
    if (delta < 1e-15) break;
  }
  cm_store(v, mu, vh, i, X);
}

// Staggered phase (and time boundary) of the link of length hop in direction mu at c.
__device__ __forceinline__ double lp_sign(const GqGeo &g, const int c[4], int mu, int hop, int apbc) {
  double s = 1;
  if (mu == 0) s = (c[3] & 1) ? -1 : 1;
  else if (mu == 1) s = ((c[3] + c[0]) & 1) ? -1 : 1;
  else if (mu == 2) s = ((c[3] + c[0] + c[1]) & 1) ? -1 : 1;
  if (mu == 3 && apbc && c[3] + hop >= g.L[3]) s = -s;
  return s;
}

// The phased link pair of direction mu at half-site i of parity cb: u[0..8]
// the forward link s fwd(x), u[9..17] MILC's back link -s' fwd(x - hop mu)^dag,
// rounded to the handle's type; f: the unphased forward links (gauge layout).
template <typename T>
__device__ __forceinline__ void phased_pair(const double *const *f, const GqGeo &g, int i, int cb, int mu, int hop,
                                            int apbc, cplx<T> *u) {
  int c[4];
  q_coords(g, i, cb, c);
  const double sf = lp_sign(g, c, mu, hop, apbc);
  const double2 *src = reinterpret_cast<const double2 *>(f[cb]) + (size_t)(9 * mu) * (size_t)g.vh;
#pragma unroll
  for (int e = 0; e < 9; ++e) {
    const double2 v = src[(size_t)e * (size_t)g.vh + i];
    u[e] = cplx<T>{(T)(sf * v.x), (T)(sf * v.y)};
  }
  int b[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) b[k] = k == mu ? (c[k] < hop ? c[k] - hop + g.L[k] : c[k] - hop) : c[k];
  const int ib = (b[0] + g.L[0] * (b[1] + g.L[1] * (b[2] + g.L[2] * b[3]))) >> 1;
  const double sb = -lp_sign(g, b, mu, hop, apbc);
  src = reinterpret_cast<const double2 *>(f[1 - cb]) + (size_t)(9 * mu) * (size_t)g.vh;  // hop is odd
#pragma unroll
  for (int rr = 0; rr < 3; ++rr)
#pragma unroll
    for (int cc = 0; cc < 3; ++cc) {
      const double2 v = src[(size_t)(3 * cc + rr) * (size_t)g.vh + ib];
      u[9 + 3 * rr + cc] = cplx<T>{(T)(sb * v.x), (T)(-sb * v.y)};
    }
}

struct PackArgs {
  const double *fat[2], *naik[2];  // unphased forward links, parity 0 / 1
  void *dfat[2], *dlng[2];         // pairs of the handle
  uint8_t *sign[2];
  unsigned long long *worst;
  GqGeo g;
  int apbc;
};

// The long links' 12-real test (recon_error) and row-2 signs.
template <typename T> __global__ void __launch_bounds__(256) k_naik_check(const PackArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, cb = blockIdx.y;
  double worst = 0;
  if (i < a.g.vh) {
    unsigned bits = 0;
#pragma unroll 1
    for (int mu = 0; mu < 4; ++mu) {
      cplx<T> u[18];
      phased_pair<T>(a.naik, a.g, i, cb, mu, 3, a.apbc, u);
      for (int h = 0; h < 2; ++h) {  // forward, back
        bool neg;
        worst = fmax(worst, recon_error(u + 9 * h, neg));
        if (neg) bits |= 1u << (2 * mu + 1 - h);
      }
    }
    a.sign[cb][i] = (uint8_t)bits;
  }
  for (int off = 32; off > 0; off >>= 1) worst = fmax(worst, __shfl_down(worst, off, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(a.worst, (unsigned long long)__double_as_longlong(worst));
}

// Fat and long pairs of both parities into the handle's tile-major chunks (NCL
// complex elements stored per long link).  Lanes run over consecutive sites:
// every load and store is one contiguous wavefront access.
template <typename T, int NCL> __global__ void __launch_bounds__(256) k_links_pack(const PackArgs a) {
  const int slot = gq_slot();
  const int v = slot % 16, mu = v & 3, cb = (v >> 2) & 1, lng = v >> 3;
  const int i = (slot / 16) * 256 + (int)threadIdx.x;
  if (i >= a.g.vh) return;
  using V = typename vec16<T>::type;
  constexpr int CPV = vec16<T>::ncplx;
  cplx<T> u[18];
  phased_pair<T>(lng ? a.naik : a.fat, a.g, i, cb, mu, lng ? 3 : 1, a.apbc, u);
  V *dst = reinterpret_cast<V *>(lng ? a.dlng[cb] : a.dfat[cb]);
  auto put = [&](int nc, auto at) {
#pragma unroll
    for (int k = 0; k < nc / CPV; ++k) {
      V w;
      if constexpr (CPV == 1) w = V{u[at(k)].re, u[at(k)].im};
      else w = V{u[at(2 * k)].re, u[at(2 * k)].im, u[at(2 * k + 1)].re, u[at(2 * k + 1)].im};
      dst[link_chunk(mu, k, i, nc / CPV)] = w;
    }
  };
  if (lng) put(2 * NCL, [](int k) { return k < NCL ? k : 9 + k - NCL; });
  else put(18, [](int k) { return k; });
}

// One level: the fat (and, with naik non-null, Naik) fields of the links u,
// FP64 in the gauge layout.  tmp: smear_tmp_mats(nmu) * 9 * vh complex numbers.
constexpr int smear_tmp_mats(int nmu) { return 2 * nmu * (3 + 6); }

template <typename T>
static void smear_level(const T *const *u, const SmearCoef &k, double *const *fat, double *const *naik, double *tmp,
                        int nmu) {
  SmearArgs a{};
  a.g = gq_geo();
  const size_t mat = 18 * (size_t)a.g.vh;  // doubles of one matrix per half-site
  for (int cb = 0; cb < 2; ++cb) {
    a.u[cb] = u[cb];
    a.m[cb] = tmp + (size_t)cb * (9 * nmu) * mat;
    a.n[cb] = a.m[cb] + (size_t)(3 * nmu) * mat;
    a.fat[cb] = fat[cb];
    a.naik[cb] = naik ? naik[cb] : nullptr;
  }
  a.k = k;
  a.nmu = nmu;
  a.lep = k.cl != 0;
  a.five = k.c5 != 0 || k.c7 != 0;
  // whole site blocks per XCD; z-regions (gq_site) where they tile the blocks exactly
  const int nbx = (a.g.vh + 255) / 256, nbp = (nbx + 7) / 8 * 8;
  a.g.zreg = a.g.L[2] % 8 == 0 && a.g.vh % 256 == 0 && nbx == nbp ? 1 : 0;
  for (a.mu0 = 0; a.mu0 < 4; a.mu0 += nmu) {
    if (a.five)
      hipLaunchKernelGGL(k_smear_inner<T>, dim3((unsigned)(6 * nmu * nbp)), dim3(256), 0, ctx().stream, a);
    hipLaunchKernelGGL(k_smear_mid<T>, dim3((unsigned)(6 * nmu * nbp)), dim3(256), 0, ctx().stream, a);
    hipLaunchKernelGGL(k_smear_outer<T>, dim3((unsigned)(2 * nmu * nbp)), dim3(256), 0, ctx().stream, a);
  }
  HIP_CHECK(hipGetLastError());
}

constexpr size_t LP_TOGETHER = (size_t)4 << 30;  // most scratch of four directions together

static double lp_now() {
  using namespace std::chrono;
  return duration<double>(steady_clock::now().time_since_epoch()).count();
}

// flags bit 0: periodic time boundary (default antiperiodic).
template <typename T>
static typename Handles<T>::L *links_from_gauge(QPHIX_info_t *info, GaugeT<T> *G, const SmearCoef &c, bool hisq,
                                                int flags) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called: links from gauge field", nullptr);
  QPHIX_REQUIRE(info && G, "links from gauge field: null argument", nullptr);
  info->status = QPHIX_FAIL;
  QPHIX_REQUIRE(G->u[0] && G->u[1], "links from gauge field: the gauge field holds no links", nullptr);
  const double t0 = lp_now();
  const int vh = ctx().g.vh;
  const size_t mat = 18 * (size_t)vh;  // doubles of one matrix per half-site
  const size_t nfield = 8 * mat;  // one field: 4 directions, both parities
  auto need = [&](int nmu) { return sizeof(double) * ((hisq ? 3 : 2) * nfield + smear_tmp_mats(nmu) * mat); };
  // All four directions run together where their scratch fits LP_TOGETHER: their
  // passes share the links of a site block in L2 (whole call, 24^4 5.8 -> 5.3 ms,
  // 16^4 1.98 -> 1.79 ms, 8^4 0.63 -> 0.46 ms, against one direction at a time).
  // Freed scratch is a kept block (context.hip) like any other: there for the next
  // call (at 24^4 a fresh allocation took up to 40 ms a call against 4 ms of
  // kernels), and given back when memory runs out.
  int nmu = 4;
  double *buf = need(4) <= LP_TOGETHER ? (double *)dev_try_alloc(need(4)) : nullptr;
  if (!buf) {
    nmu = 1;
    buf = (double *)dev_alloc(need(1));
  }
  unsigned long long *dmax = (unsigned long long *)dev_alloc(sizeof(unsigned long long));
  auto *L = new typename Handles<T>::L;
  L->parity = QPHIX_EVENODD;
  auto bail = [&]() -> typename Handles<T>::L * {  // an allocation failed, error recorded
    HIP_CHECK(hipStreamSynchronize(ctx().stream));
    links_free<T>(L);
    delete L;
    dev_free(dmax);
    dev_free(buf);
    info->status = QPHIX_MEM_ERROR;
    return nullptr;
  };
  if (!buf || !dmax) return bail();
  double *fat[2] = {buf, buf + 4 * mat}, *naik[2] = {buf + nfield, buf + nfield + 4 * mat};
  double *tmp = buf + (hisq ? 3 : 2) * nfield;
  if (hisq) {
    // level 1: V = fat7(U), then W = unitary polar factor of V
    double *w[2] = {buf + 2 * nfield, buf + 2 * nfield + 4 * mat};
    smear_level<T>(G->u, SmearCoef{1.0 / 8, 1.0 / 16, 1.0 / 64, 1.0 / 384, 0.0, 0.0}, w, nullptr, tmp, nmu);
    hipLaunchKernelGGL(k_u3_project, dim3((unsigned)((vh + 255) / 256), 8), dim3(256), 0, ctx().stream, w[0], w[1],
                       vh);
    // level 2 from W: fat links and the Naik links -(1 + eps)/24 W W W
    smear_level<double>(w, c, fat, naik, tmp, nmu);
  } else {
    smear_level<T>(G->u, c, fat, naik, tmp, nmu);
  }
  PackArgs a{};
  a.g = gq_geo();
  a.apbc = (flags & 1) ? 0 : 1;
  a.worst = dmax;
  for (int cb = 0; cb < 2; ++cb) {
    a.fat[cb] = fat[cb];
    a.naik[cb] = naik[cb];
  }
  const int nbx = (vh + 255) / 256;
  bool can12 = long_recon_mode() != 18;
  if (can12) {
    for (int cb = 0; cb < 2; ++cb) {
      a.sign[cb] = L->lsign[cb] = (uint8_t *)dev_alloc((size_t)vh);
      if (!L->lsign[cb]) return bail();
    }
    HIP_CHECK(hipMemsetAsync(dmax, 0, sizeof(unsigned long long), ctx().stream));
    hipLaunchKernelGGL(k_naik_check<T>, dim3((unsigned)nbx, 2), dim3(256), 0, ctx().stream, a);
    HIP_CHECK(hipGetLastError());
    double worst = 0;
    HIP_CHECK(hipMemcpyAsync(&worst, dmax, sizeof(worst), hipMemcpyDeviceToHost, ctx().stream));
    HIP_CHECK(hipStreamSynchronize(ctx().stream));
    can12 = worst <= recon_tol<T>();
  }
  for (int cb = 0; cb < 2 && !can12; ++cb) {
    dev_free(L->lsign[cb]);
    L->lsign[cb] = nullptr;
  }
  L->recon = can12 ? 12 : 18;
  for (int cb = 0; cb < 2; ++cb) {
    a.dfat[cb] = L->fat[cb] = (T *)dev_alloc(sizeof(T) * 144 * link_sites(vh));
    a.dlng[cb] = L->lng[cb] = (T *)dev_alloc(sizeof(T) * 8 * L->recon * link_sites(vh));
    if (!L->fat[cb] || !L->lng[cb]) return bail();
  }
  const dim3 pgrid((unsigned)(16 * ((nbx + 7) / 8 * 8)));
  if (can12) hipLaunchKernelGGL((k_links_pack<T, 6>), pgrid, dim3(256), 0, ctx().stream, a);
  else hipLaunchKernelGGL((k_links_pack<T, 9>), pgrid, dim3(256), 0, ctx().stream, a);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipStreamSynchronize(ctx().stream));
  dev_free(dmax);
  dev_free(buf);
  info->final_sec = lp_now() - t0;
  // the nest of every link on its own: 168 staple products and 2 Naik
  // products, 216 flops each (x 2 + the projection for HISQ)
  info->final_flop = (hisq ? 2.0 : 1.0) * 170.0 * 216.0 * 8.0 * vh;
  info->status = QPHIX_SUCCESS;
  return L;
}

} // namespace qphix

using namespace qphix;

extern "C" {

#define QPHIX_LP_API(P, T)                                                                                   \
  QPHIX_##P##3_FermionLinksAsqtad *QPHIX_##P##3_asqtad_create_L_from_G(                                      \
      QPHIX_info_t *info, const QPHIX_MI355X_asqtad_coeffs_t *coeffs, QPHIX_##P##3_GaugeField *G, int flags) { \
    QPHIX_REQUIRE(coeffs, "asqtad_create_L_from_G: null coefficients", nullptr);                             \
    const SmearCoef c{coeffs->one_link,     coeffs->three_staple, coeffs->five_staple,                      \
                      coeffs->seven_staple, coeffs->lepage,       coeffs->naik};                            \
    return static_cast<QPHIX_##P##3_FermionLinksAsqtad *>(links_from_gauge<T>(info, G, c, false, flags)); \
  }                                                                                                          \
  QPHIX_##P##3_FermionLinksAsqtad *QPHIX_##P##3_hisq_create_L_from_G(QPHIX_info_t *info,                      \
                                                                     QPHIX_##P##3_GaugeField *G,              \
                                                                     double naik_eps, int flags) {            \
    return static_cast<QPHIX_##P##3_FermionLinksAsqtad *>(                                                   \
        links_from_gauge<T>(info, G, hisq_level2(naik_eps), true, flags));                         \
  }

QPHIX_LP_API(D, double)
QPHIX_LP_API(F, float)

} // extern "C"
