// fields.hip -- create / extract / destroy for colour vectors, asqtad links,
// gauge fields and momenta; raw MILC order <-> device layouts.
//
// Reference: qphix_d3.cpp:79-174 (V), 177-343 (G), 347-488 (F), 490-559 (V out),
// 562-742 (G out), 745-949 (F out), 970-1206 (L), 1208-1245 (destroy).
// Raw arrays are even sites first, 6 (vectors) or 72 (links, momenta) reals per
// site (convention C1).  Link import keeps every slot exactly as the caller gave
// it (C4); long links are stored as 12 reals only when row 2 of every long link
// is +-conj(row0 x row1) to rounding, with the sign kept per link (1 bit),
// otherwise as 18 -- so the stored operator always equals the given one.
#include "handles.h"
#include "device.h"
#include "hostio.h"
#include "raw_tile.h"
#include "qphix_mi355x.h"

#include <algorithm>
#include <cstring>

namespace qphix {

static int g_recon_mode = 0;
int long_recon_mode() { return g_recon_mode; }

// ------------------------------------------------------------------ kernels
// The raw <-> device conversions of links work on tiles of 64 sites held in
// LDS (raw_tile.h): whole-line accesses on both sides, and 28 blocks or more
// for the few thousand sites of a transfer's chunk.

__device__ __forceinline__ void atomic_max_nonneg(unsigned long long *a, double v) {
  atomicMax(a, (unsigned long long)__double_as_longlong(v));
}

// Sites [first, first + n) of the raw link blocks fwd (blockIdx.y = 0) and back
// (1), site first at their beginnings, into the pairs of dst, ncl complex
// elements of each link.  sign non-null: also the 12-real test (recon_error,
// largest into *maxbits) and row-2 signs (sign zeroed beforehand).
template <typename T>
__global__ void __launch_bounds__(256) k_import_pairs(T *dst, const T *fwd, const T *back, int first, int ncl,
                                                      uint8_t *sign, unsigned long long *maxbits) {
  __shared__ __align__(16) T tile[RAW_TILE_REALS];
  const int h = blockIdx.y, base = blockIdx.x * 64;
  raw_tile_in<T>(tile, (h ? back : fwd) + 72 * (size_t)base);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = first + base + lane;
  const cplx<T> *mine = reinterpret_cast<const cplx<T> *>(tile + RAW_TILE_STRIDE * lane);
  if (sign) {  // one link per work-item: direction = wave
    bool neg;
    double worst = recon_error(mine + 9 * wave, neg);
    // bit 2 mu + 1 forward, 2 mu back, in the byte of site i
    if (neg) atomicOr(reinterpret_cast<unsigned *>(sign) + i / 4, 1u << (8 * (i % 4) + 2 * wave + 1 - h));
    for (int off = 32; off > 0; off >>= 1) worst = fmax(worst, __shfl_down(worst, off, 64));
    if (lane == 0) atomic_max_nonneg(maxbits, worst);
  }
  constexpr int CPV = vec16<T>::ncplx;
  cplx<T> *d = reinterpret_cast<cplx<T> *>(dst);
  for (int q = wave; q < 4 * ncl; q += 4) {
    const int mu = q / ncl, kk = q % ncl, k = h * ncl + kk;
    d[link_chunk(mu, k / CPV, i, 2 * ncl / CPV) * CPV + k % CPV] = mine[9 * mu + kk];
  }
}

// Forward links of the sites [first, first + n) back to raw order (extract_L):
// blockIdx.y = 0 fat, 1 long; 12-stored long links get their third row rebuilt
// with the stored sign.
template <typename T>
__global__ void __launch_bounds__(256) k_export_fwd(const T *fat, const T *lng, const uint8_t *sign, int first, int ncl,
                                                    T *fat_raw, T *lng_raw) {
  __shared__ __align__(16) T tile[RAW_TILE_REALS];
  const int base = blockIdx.x * 64, lane = threadIdx.x & 63, mu = threadIdx.x >> 6;
  const int i = first + base + lane;
  constexpr int CPV = vec16<T>::ncplx;
  const bool isl = blockIdx.y != 0;
  const int nc = isl ? ncl : 9;
  const cplx<T> *src = reinterpret_cast<const cplx<T> *>(isl ? lng : fat);
  cplx<T> *mine = reinterpret_cast<cplx<T> *>(tile + RAW_TILE_STRIDE * lane) + 9 * mu;
  cplx<double> w[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    if (k >= nc) break;
    const cplx<T> v = src[link_chunk(mu, k / CPV, i, 2 * nc / CPV) * CPV + k % CPV];
    w[k] = cplx<double>{(double)v.re, (double)v.im};
  }
  if (nc == 6) recon_row2(w, ((sign[i] >> (2 * mu + 1)) & 1u) ? -1.0 : 1.0);
#pragma unroll
  for (int k = 0; k < 9; ++k) mine[k] = cplx<T>{(T)w[k].re, (T)w[k].im};
  raw_tile_out<T>((isl ? lng_raw : fat_raw) + 72 * (size_t)base, tile);
}

// Load complex k (row-major) of the forward (fb=1) or back (fb=0) link of
// direction mu at site i.
template <typename T>
__device__ __forceinline__ cplx<double> link_elem(const T *base, int vh, int ncl, int mu, int fb,
                                                  int k, int i) {
  constexpr int CPV = vec16<T>::ncplx;
  const int kk = fb ? k : ncl + k;
  const size_t chunk = link_chunk(mu, kk / CPV, i, 2 * ncl / CPV);
  const T *s = base + chunk * (2 * CPV) + 2 * (kk % CPV);
  return cplx<double>{(double)s[0], (double)s[1]};
}

template <typename T>
__device__ void load_link(const T *base, const uint8_t *sign, int vh, int ncl, int mu, int fb,
                          int i, cplx<double> *w) {
  for (int k = 0; k < ncl; ++k) w[k] = link_elem(base, vh, ncl, mu, fb, k, i);
  if (ncl == 6) recon_row2(w, ((sign[i] >> (2 * mu + fb)) & 1u) ? -1.0 : 1.0);
}

// max |back_mu(x) -/+ U_mu(x - hop)^dagger| for fat (hop 1) and long (hop 3).
template <typename T>
__global__ void k_backcheck(const T *fat_c, const T *lng_c, const uint8_t *sgn_c, const T *fat_o,
                            const T *lng_o, const uint8_t *sgn_o, int ncl, Geo g, int cb,
                            unsigned long long *out4) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double m[4] = {0, 0, 0, 0};
  if (i < g.vh) {
    SiteNbr n;
    site_neighbours(g, i, cb, n);
    for (int mu = 0; mu < 4; ++mu)
      for (int kind = 0; kind < 2; ++kind) {
        cplx<double> b[9], u[9];
        if (kind == 0) {
          load_link(fat_c, nullptr, g.vh, 9, mu, 0, i, b);
          load_link(fat_o, nullptr, g.vh, 9, mu, 1, n.b1[mu], u);
        } else {
          load_link(lng_c, sgn_c, g.vh, ncl, mu, 0, i, b);
          load_link(lng_o, sgn_o, g.vh, ncl, mu, 1, n.b3[mu], u);
        }
        for (int r = 0; r < 3; ++r)
          for (int c = 0; c < 3; ++c) {
            const cplx<double> a{u[3 * c + r].re, -u[3 * c + r].im};  // adj(u)[r][c]
            const cplx<double> x = b[3 * r + c];
            m[2 * kind] = fmax(m[2 * kind], fmax(fabs(x.re + a.re), fabs(x.im + a.im)));
            m[2 * kind + 1] = fmax(m[2 * kind + 1], fmax(fabs(x.re - a.re), fabs(x.im - a.im)));
          }
      }
  }
  for (int k = 0; k < 4; ++k) {
    double v = m[k];
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    if ((threadIdx.x & 63) == 0) atomic_max_nonneg(out4 + k, v);
  }
}

// FP64 chunk layout -> FP32 chunk layout (same pairs, same recon).
__global__ void k_links_to_float(float *dst, const double *src, int vh, int nc_pair) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  for (int mu = 0; mu < 4; ++mu)
    for (int k = 0; k < nc_pair; ++k) {
      const double *s = src + link_chunk(mu, k, i, nc_pair) * 2;
      float *d = dst + link_chunk(mu, k / 2, i, nc_pair / 2) * 4 + 2 * (k % 2);
      d[0] = (float)s[0];
      d[1] = (float)s[1];
    }
}

// tan(arg z / 2) for the 8-real form (recon8), from the half-angle identities
// tan(t/2) = sin t / (1 + cos t) = (1 - cos t) / sin t, each used where it does
// not cancel; arg z = pi maps to 1e18 (phase -1 to FP32 rounding), z = 0 to 0.
__device__ double half_tan(double x, double y) {
  const double r = hypot(x, y);
  if (r == 0) return 0;
  const double h = x >= 0 ? y / (r + x) : (y == 0 ? 1e18 : (r - x) / y);
  return fmin(fmax(h, -1e18), 1e18);
}

// FP64 12-real long links -> FP32 8-real form: per link U01, U02, U10 and the
// half-angle tangents of U00 and U20 = s conj(U01 U12 - U02 U11) (s the stored
// row-2 sign).  The 8-real rebuild takes |U00| and |U20| from unitarity, so a
// link has no usable 8-real form when its rows 0 and 1 are not orthonormal to
// 1e-6 (the 12-real check only ties row 2 to them) or n = |U01|^2 + |U02|^2 <
// 1e-10; such links are counted in *bad and the caller keeps the 12-real form.
__global__ void k_links_to_float8(float *dst, const double *src, const uint8_t *sign, int vh,
                                  unsigned *bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  unsigned nbad = 0;
  for (int mu = 0; mu < 4; ++mu)
    for (int fb = 0; fb < 2; ++fb) {  // fb 0: forward link (chunks 0-5), 1: back link (6-11)
      double u[12];
      for (int k = 0; k < 6; ++k) {
        const double *c = src + link_chunk(mu, 6 * fb + k, i, 12) * 2;
        u[2 * k] = c[0];
        u[2 * k + 1] = c[1];
      }
      const double s = ((sign[i] >> (2 * mu + (fb ? 0 : 1))) & 1u) ? -1.0 : 1.0;
      // U01 U12 - U02 U11
      const double xr = u[2] * u[10] - u[3] * u[11] - (u[4] * u[8] - u[5] * u[9]);
      const double xi = u[2] * u[11] + u[3] * u[10] - (u[4] * u[9] + u[5] * u[8]);
      const double n = u[2] * u[2] + u[3] * u[3] + u[4] * u[4] + u[5] * u[5];
      const double n0 = u[0] * u[0] + u[1] * u[1] + n;
      const double n1 = u[6] * u[6] + u[7] * u[7] + u[8] * u[8] + u[9] * u[9] + u[10] * u[10] + u[11] * u[11];
      double dr = 0, di = 0;  // row 0 . conj(row 1)
      for (int c = 0; c < 3; ++c) {
        dr += u[2 * c] * u[6 + 2 * c] + u[2 * c + 1] * u[6 + 2 * c + 1];
        di += u[2 * c + 1] * u[6 + 2 * c] - u[2 * c] * u[6 + 2 * c + 1];
      }
      if (!(n >= 1e-10) || !(fabs(n0 - 1) <= 1e-6) || !(fabs(n1 - 1) <= 1e-6) || !(hypot(dr, di) <= 1e-6)) ++nbad;
      const float v[8] = {(float)u[2], (float)u[3], (float)u[4], (float)u[5], (float)u[6], (float)u[7],
                          (float)half_tan(u[0], u[1]), (float)half_tan(s * xr, -s * xi)};
      for (int k = 0; k < 4; ++k) {
        float *d = dst + link_chunk(mu, (4 * fb + k) / 2, i, 4) * 4 + 2 * (k % 2);
        d[0] = v[2 * k];
        d[1] = v[2 * k + 1];
      }
    }
  if (nbad) atomicAdd(bad, nbad);
}

// FP64 links (double2 chunks) -> 16-bit fixed point (Q16 chunks), per site
// and direction one pair of nc_pair complex elements (forward link, then back
// link), each link with its own scale.
__global__ void k_links_to_q16(uint4 *dst, const double *src, int vh, int nc_pair) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  const int nch = nc_pair == 12 ? link_nch<Q16>(12) : link_nch<Q16>(18);
  for (int mu = 0; mu < 4; ++mu) {
    double x[36];
    for (int k = 0; k < nc_pair; ++k) {
      const double *c = src + link_chunk(mu, k, i, nc_pair) * 2;
      x[2 * k] = c[0];
      x[2 * k + 1] = c[1];
    }
    float sc[2];
    for (int h = 0; h < 2; ++h) {
      double m = 0;
      for (int e = h * nc_pair; e < (h + 1) * nc_pair; ++e) m = fmax(m, fabs(x[e]));
      float f = (float)m;
      if ((double)f < m) f = nextafterf(f, INFINITY);  // |x| / f <= 1
      sc[h] = f;
    }
    unsigned w[20] = {};
    for (int e = 0; e < 2 * nc_pair; ++e) {
      const float f = sc[e < nc_pair ? 0 : 1];
      int q = f > 0.f ? (int)rint(x[e] / (double)f * 32767.0) : 0;
      q = q > 32767 ? 32767 : (q < -32767 ? -32767 : q);
      w[e / 2] |= ((unsigned)q & 0xffffu) << (16 * (e % 2));
    }
    w[4 * nch - 2] = __float_as_uint(sc[0]);
    w[4 * nch - 1] = __float_as_uint(sc[1]);
    for (int k = 0; k < nch; ++k)
      dst[link_chunk(mu, k, i, nch)] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
  }
}

// Momentum raw (anti-Hermitian A, 18 reals) -> 8 reals of H = -iA
// (qphix_d3.cpp:420-433): [ReH01, ImH01, ReH02, ImH02, ReH12, ImH12, H00, H11].
template <typename T> __global__ void k_mom_in(T *h, const T *raw, int nlinks) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= nlinks) return;
  const T *a = raw + 18 * (size_t)l;
  T *o = h + 8 * (size_t)l;
  // H_rc = -i A_rc : Re H = Im A, Im H = -Re A
  o[0] = a[2 * 1 + 1];   o[1] = -a[2 * 1];        // (0,1)
  o[2] = a[2 * 2 + 1];   o[3] = -a[2 * 2];        // (0,2)
  o[4] = a[6 + 2 * 2 + 1]; o[5] = -a[6 + 2 * 2];  // (1,2)
  o[6] = a[1];           o[7] = a[6 + 2 * 1 + 1]; // ImA00, ImA11
}

// Inverse (qphix_d3.cpp:809-842): A = iH, Re A_kk = 0, Im A22 = -Im A00 - Im A11.
template <typename T> __global__ void k_mom_out(T *raw, const T *h, int nlinks) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= nlinks) return;
  const T *o = h + 8 * (size_t)l;
  T *a = raw + 18 * (size_t)l;
  const int pr[3][2] = {{0, 1}, {0, 2}, {1, 2}};
  for (int q = 0; q < 3; ++q) {
    const int r = pr[q][0], c = pr[q][1];
    const T hr = o[2 * q], hi = o[2 * q + 1];
    a[6 * r + 2 * c] = -hi;  // A_rc = i H_rc
    a[6 * r + 2 * c + 1] = hr;
    a[6 * c + 2 * r] = hi;   // A_cr = -conj(A_rc)
    a[6 * c + 2 * r + 1] = hr;
  }
  a[0] = 0; a[1] = o[6];
  a[8] = 0; a[9] = o[7];
  a[16] = 0; a[17] = -o[6] - o[7];
}

// ------------------------------------------------------------------ helpers
static inline int nblk(int n, int b = 256) { return (n + b - 1) / b; }

static inline void d2h(void *h, const void *d, size_t bytes) {
  HIP_CHECK(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, ctx().stream));
}
static inline void sync() { HIP_CHECK(hipStreamSynchronize(ctx().stream)); }

template <typename T> void links_free(LinksT<T> *L) {
  if (!L) return;
  for (int cb = 0; cb < 2; ++cb) {
    dev_free(L->fat[cb]);
    dev_free(L->lng[cb]);
    dev_free(L->lsign[cb]);
    L->fat[cb] = L->lng[cb] = nullptr;
    L->lsign[cb] = nullptr;
  }
  if (L->sloppy) {
    links_free(L->sloppy);
    delete L->sloppy;
    L->sloppy = nullptr;
  }
  if (L->sloppy16) {
    links_free(L->sloppy16);
    delete L->sloppy16;
    L->sloppy16 = nullptr;
  }
  if (L->sloppy8) {
    links_free(L->sloppy8);
    delete L->sloppy8;
    L->sloppy8 = nullptr;
  }
}
template void links_free<double>(LinksT<double> *);
template void links_free<float>(LinksT<float> *);
template void links_free<Q16>(LinksT<Q16> *);

bool links_to_float(const LinksT<double> &Ld, LinksT<float> &Lf) {
  const int vh = ctx().g.vh;
  Lf.recon = Ld.recon;
  Lf.parity = Ld.parity;
  for (int cb = 0; cb < 2; ++cb) {
    if (!Ld.fat[cb]) continue;
    Lf.fat[cb] = (float *)dev_alloc(sizeof(float) * 4 * 36 * link_sites(vh));
    Lf.lng[cb] = (float *)dev_alloc(sizeof(float) * 4 * 2 * Ld.recon * link_sites(vh));
    if (Ld.lsign[cb]) Lf.lsign[cb] = (uint8_t *)dev_alloc((size_t)vh);
    if (!Lf.fat[cb] || !Lf.lng[cb] || (Ld.lsign[cb] && !Lf.lsign[cb])) {  // error recorded
      HIP_CHECK(hipStreamSynchronize(ctx().stream));  // earlier parity's copies done
      links_free(&Lf);
      return false;
    }
    hipLaunchKernelGGL(k_links_to_float, dim3(nblk(vh)), dim3(256), 0, ctx().stream, Lf.fat[cb],
                       Ld.fat[cb], vh, 18);
    hipLaunchKernelGGL(k_links_to_float, dim3(nblk(vh)), dim3(256), 0, ctx().stream, Lf.lng[cb],
                       Ld.lng[cb], vh, Ld.recon == 12 ? 12 : 18);
    if (Ld.lsign[cb])
      HIP_CHECK(hipMemcpyAsync(Lf.lsign[cb], Ld.lsign[cb], (size_t)vh, hipMemcpyDeviceToDevice,
                               ctx().stream));
  }
  HIP_CHECK(hipGetLastError());
  return true;
}

// FP32 copy with 8-real long links (fat links as links_to_float).  Returns 0 on
// success, 1 when some long link has no 8-real form (nothing kept, no error),
// -1 when out of device memory (error recorded).
static int links_to_float8(const LinksT<double> &Ld, LinksT<float> &Lf) {
  const int vh = ctx().g.vh;
  Lf.recon = 8;
  Lf.parity = Ld.parity;
  unsigned *bad = (unsigned *)dev_alloc(sizeof(unsigned));
  if (!bad) return -1;
  HIP_CHECK(hipMemsetAsync(bad, 0, sizeof(unsigned), ctx().stream));
  for (int cb = 0; cb < 2; ++cb) {
    if (!Ld.fat[cb]) continue;
    Lf.fat[cb] = (float *)dev_alloc(sizeof(float) * 4 * 36 * link_sites(vh));
    Lf.lng[cb] = (float *)dev_alloc(sizeof(float) * 4 * 2 * 8 * link_sites(vh));
    Lf.lsign[cb] = (uint8_t *)dev_alloc((size_t)vh);
    if (!Lf.fat[cb] || !Lf.lng[cb] || !Lf.lsign[cb]) {  // error recorded
      HIP_CHECK(hipStreamSynchronize(ctx().stream));
      links_free(&Lf);
      dev_free(bad);
      return -1;
    }
    hipLaunchKernelGGL(k_links_to_float, dim3(nblk(vh)), dim3(256), 0, ctx().stream, Lf.fat[cb],
                       Ld.fat[cb], vh, 18);
    hipLaunchKernelGGL(k_links_to_float8, dim3(nblk(vh)), dim3(256), 0, ctx().stream, Lf.lng[cb],
                       Ld.lng[cb], Ld.lsign[cb], vh, bad);
    HIP_CHECK(hipMemcpyAsync(Lf.lsign[cb], Ld.lsign[cb], (size_t)vh, hipMemcpyDeviceToDevice, ctx().stream));
  }
  HIP_CHECK(hipGetLastError());
  unsigned nbad = 0;
  HIP_CHECK(hipMemcpyAsync(&nbad, bad, sizeof(unsigned), hipMemcpyDeviceToHost, ctx().stream));
  HIP_CHECK(hipStreamSynchronize(ctx().stream));
  dev_free(bad);
  if (nbad) {
    links_free(&Lf);
    return 1;
  }
  return 0;
}

bool links_to_q16(const LinksT<double> &Ld, LinksT<Q16> &Lq) {
  const int vh = ctx().g.vh;
  Lq.recon = Ld.recon;
  Lq.parity = Ld.parity;
  const int ncl = Ld.recon == 12 ? 12 : 18;
  for (int cb = 0; cb < 2; ++cb) {
    if (!Ld.fat[cb]) continue;
    Lq.fat[cb] = (Q16 *)dev_alloc(16 * 4 * (size_t)link_nch<Q16>(18) * link_sites(vh));
    Lq.lng[cb] = (Q16 *)dev_alloc(16 * 4 * (size_t)link_nch<Q16>(ncl) * link_sites(vh));
    if (Ld.lsign[cb]) Lq.lsign[cb] = (uint8_t *)dev_alloc((size_t)vh);
    if (!Lq.fat[cb] || !Lq.lng[cb] || (Ld.lsign[cb] && !Lq.lsign[cb])) {  // error recorded
      HIP_CHECK(hipStreamSynchronize(ctx().stream));  // earlier parity's copies done
      links_free(&Lq);
      return false;
    }
    hipLaunchKernelGGL(k_links_to_q16, dim3(nblk(vh)), dim3(256), 0, ctx().stream,
                       reinterpret_cast<uint4 *>(Lq.fat[cb]), Ld.fat[cb], vh, 18);
    hipLaunchKernelGGL(k_links_to_q16, dim3(nblk(vh)), dim3(256), 0, ctx().stream,
                       reinterpret_cast<uint4 *>(Lq.lng[cb]), Ld.lng[cb], vh, ncl);
    if (Ld.lsign[cb])
      HIP_CHECK(hipMemcpyAsync(Lq.lsign[cb], Ld.lsign[cb], (size_t)vh, hipMemcpyDeviceToDevice,
                               ctx().stream));
  }
  HIP_CHECK(hipGetLastError());
  return true;
}

const LinksT<float> *sloppy_links(LinksT<double> *L) {
  if (!L->sloppy) {
    auto *s = new LinksT<float>;
    if (!links_to_float(*L, *s)) {
      delete s;
      return nullptr;
    }
    L->sloppy = s;
  }
  return L->sloppy;
}

static int g_sloppy_long_recon = 8;

// The FP32 links of the mixed solver's sloppy operator: long links in their
// 8-real form when set (the default), the FP64 links keep 12 reals and every
// long link has that form; otherwise the FP32 copy of sloppy_links.
const LinksT<float> *sloppy_links_solver(LinksT<double> *L) {
  if (g_sloppy_long_recon == 8 && L->recon == 12 && !L->no8) {
    if (!L->sloppy8) {
      auto *s = new LinksT<float>;
      const int rc = links_to_float8(*L, *s);
      if (rc < 0) {
        delete s;
        return nullptr;
      }
      if (rc == 0) L->sloppy8 = s;
      else {
        delete s;
        L->no8 = true;
      }
    }
    if (L->sloppy8) return L->sloppy8;
  }
  return sloppy_links(L);
}

const LinksT<Q16> *sloppy_links16(LinksT<double> *L) {
  if (!L->sloppy16) {
    auto *s = new LinksT<Q16>;
    if (!links_to_q16(*L, *s)) {
      delete s;
      return nullptr;
    }
    L->sloppy16 = s;
  }
  return L->sloppy16;
}

static int g_sloppy_link_bits = 32;
int sloppy_link_bits() { return g_sloppy_link_bits; }

// ------------------------------------------------------------------ V
// Raw MILC order [site][colour][re, im] <-> the tile-major spinor storage
// (Spin<T>), one work-item per site of [first, first + n) of one parity.
template <typename T> __global__ void k_spin_from_raw(T *dst, const T *raw, int first, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  cplx<T> v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = cplx<T>{raw[6 * (size_t)i + 2 * c], raw[6 * (size_t)i + 2 * c + 1]};
  Spin<T>::store(dst, first + i, v);
}

template <typename T> __global__ void k_spin_to_raw(T *raw, const T *src, int first, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  cplx<T> v[3];
  Spin<T>::load(src, first + i, v);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    raw[6 * (size_t)i + 2 * c] = v[c].re;
    raw[6 * (size_t)i + 2 * c + 1] = v[c].im;
  }
}

// The transfer of the parities in `evenodd` of a raw array with `reals` reals a
// site: where it begins, and how many halves it has.
struct RawHalves {
  int first, n;  // first parity, number of parities
  explicit RawHalves(int evenodd)
      : first(evenodd & QPHIX_EVEN ? 0 : 1), n(!!(evenodd & QPHIX_EVEN) + !!(evenodd & QPHIX_ODD)) {}
  template <typename T> HostArray array(const T *p, size_t reals) const {
    return HostArray{reinterpret_cast<char *>(const_cast<T *>(p + first * reals * (size_t)ctx().g.vh)),
                     reals * sizeof(T)};
  }
  // parity of a chunk and its first site within it
  int parity(size_t site) const { return first + (site >= (size_t)ctx().g.vh ? 1 : 0); }
  static int local(size_t site) { return (int)(site % (size_t)ctx().g.vh); }
};

// qphix_d3.cpp:79-174 (create_V): the raw half of each requested parity is
// copied to the device and reordered there.
template <typename T>
static typename Handles<T>::V *create_V(const T *src, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:create_V", nullptr);
  const int vh = ctx().g.vh;
  const size_t nv = 6 * (size_t)vh;
  char *stage = nullptr;
  if (src) {
    stage = (char *)dev_alloc(host_stage_bytes(6 * sizeof(T), vh, std::max(RawHalves(evenodd).n, 1)));
    if (!stage) return nullptr;  // error recorded
  }
  auto *V = new typename Handles<T>::V;
  V->parity = evenodd;
  for (int cb = 0; cb < 2; ++cb) {
    const int bit = cb ? QPHIX_ODD : QPHIX_EVEN;
    if (!(evenodd & bit)) continue;
    V->half[cb] = (T *)dev_alloc(sizeof(T) * nv);
    if (!V->half[cb]) {  // dev_alloc has recorded the error
      dev_free(V->half[0]);
      dev_free(V->half[1]);
      dev_free(stage);
      delete V;
      return nullptr;
    }
    if (!src) HIP_CHECK(hipMemsetAsync(V->half[cb], 0, sizeof(T) * nv, ctx().stream));
  }
  if (src) {
    const RawHalves rh(evenodd);
    const HostArray a = rh.array(src, 6);
    host_to_device(&a, 1, vh, rh.n, stage, [&](char *const *d, size_t first, size_t n) {
      hipLaunchKernelGGL(k_spin_from_raw<T>, dim3(nblk((int)n)), dim3(256), 0, ctx().stream,
                         V->half[rh.parity(first)], (const T *)d[0], rh.local(first), (int)n);
      HIP_CHECK(hipGetLastError());
    });
  } else {
    sync();
  }
  dev_free(stage);
  return V;
}

// The parities written are those the vector holds (src->parity), as in the
// reference (qphix_d3.cpp:495-553 ignores the evenodd argument).
template <typename T> static void extract_V(T *dest, const typename Handles<T>::V *V) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:extract_V");
  QPHIX_REQUIRE(V && dest, "extract_V: null argument");
  const int vh = ctx().g.vh;
  const RawHalves rh((V->half[0] ? QPHIX_EVEN : 0) | (V->half[1] ? QPHIX_ODD : 0));
  if (rh.n == 0) return;
  char *stage = (char *)dev_alloc(host_stage_bytes(6 * sizeof(T), vh, rh.n));
  if (!stage) return;  // error recorded
  const HostArray a = rh.array(dest, 6);
  device_to_host(&a, 1, vh, rh.n, stage, [&](char *const *d, size_t first, size_t n) {
    hipLaunchKernelGGL(k_spin_to_raw<T>, dim3(nblk((int)n)), dim3(256), 0, ctx().stream, (T *)d[0],
                       V->half[rh.parity(first)], rh.local(first), (int)n);
    HIP_CHECK(hipGetLastError());
  });
  dev_free(stage);
}

template <typename T> static void destroy_V(typename Handles<T>::V *V) {
  if (!V) return;
  if (ctx().initialised) HIP_CHECK(hipStreamSynchronize(ctx().stream));
  dev_free(V->half[0]);
  dev_free(V->half[1]);
  delete V;
}

// ------------------------------------------------------------------ L
// Links from the caller's raw arrays, each read once.  The Naik links are
// stored as 12 reals while every one seen is SU(3) times a sign (k_import_pairs;
// looked at after the first chunk, where scaled links already show, and at the
// end); when one is not, they are read again into 18.
template <typename T>
static typename Handles<T>::L *create_L(const T *fat, const T *lng, const T *fatback,
                                        const T *lngback, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:create_L", nullptr);
  QPHIX_REQUIRE(fat && lng && fatback && lngback, "create_L: null link array", nullptr);
  const int vh = ctx().g.vh;
  const RawHalves rh(evenodd);
  auto *L = new typename Handles<T>::L;
  L->parity = evenodd;
  char *stage = (char *)dev_alloc(host_stage_bytes(4 * 72 * sizeof(T), vh, std::max(rh.n, 1)));
  unsigned long long *dmax = (unsigned long long *)dev_alloc(sizeof(unsigned long long) * 4);
  auto done = [&](bool ok) -> typename Handles<T>::L * {
    sync();
    dev_free(stage);
    dev_free(dmax);
    if (ok) return L;
    links_free<T>(L);
    delete L;
    return nullptr;
  };
  if (!stage || !dmax) return done(false);
  auto wanted = [&](int cb) { return (evenodd & (cb ? QPHIX_ODD : QPHIX_EVEN)) != 0; };
  // storage of the long links: 12 (with signs) or 18 reals; false: error recorded
  auto alloc_long = [&](int recon) {
    L->recon = recon;
    for (int cb = 0; cb < 2; ++cb) {
      if (!wanted(cb)) continue;
      if (recon == 12) {
        if (!(L->lsign[cb] = (uint8_t *)dev_alloc((size_t)vh))) return false;
        HIP_CHECK(hipMemsetAsync(L->lsign[cb], 0, (size_t)vh, ctx().stream));
      }
      if (!(L->lng[cb] = (T *)dev_alloc(sizeof(T) * 8 * recon * link_sites(vh)))) return false;
    }
    return true;
  };
  auto drop_long = [&]() {
    sync();
    for (int cb = 0; cb < 2; ++cb) {
      dev_free(L->lng[cb]);
      dev_free(L->lsign[cb]);
      L->lng[cb] = nullptr;
      L->lsign[cb] = nullptr;
    }
  };
  auto all12 = [&]() {
    unsigned long long bits = 0;
    d2h(&bits, dmax, sizeof(bits));
    sync();
    double worst;
    std::memcpy(&worst, &bits, sizeof(worst));
    return worst <= recon_tol<T>();
  };
  auto put_long = [&](int cb, const char *f, const char *b, int first, size_t n) {
    hipLaunchKernelGGL(k_import_pairs<T>, dim3((unsigned)(n / 64), 2), dim3(256), 0, ctx().stream, L->lng[cb],
                       (const T *)f, (const T *)b, first, L->recon == 12 ? 6 : 9, L->lsign[cb], dmax);
    HIP_CHECK(hipGetLastError());
  };
  HIP_CHECK(hipMemsetAsync(dmax, 0, sizeof(unsigned long long), ctx().stream));
  for (int cb = 0; cb < 2; ++cb)
    if (wanted(cb) && !(L->fat[cb] = (T *)dev_alloc(sizeof(T) * 144 * link_sites(vh)))) return done(false);
  if (!alloc_long(long_recon_mode() != 18 ? 12 : 18)) return done(false);
  bool looked = L->recon == 18, ok = true;
  const HostArray a[4] = {rh.array(fat, 72), rh.array(fatback, 72), rh.array(lng, 72), rh.array(lngback, 72)};
  host_to_device(a, 4, vh, rh.n, stage, [&](char *const *d, size_t site, size_t n) {
    if (!ok) return;
    const int cb = rh.parity(site), first = rh.local(site);
    hipLaunchKernelGGL(k_import_pairs<T>, dim3((unsigned)(n / 64), 2), dim3(256), 0, ctx().stream, L->fat[cb],
                       (const T *)d[0], (const T *)d[1], first, 9, (uint8_t *)nullptr, (unsigned long long *)nullptr);
    put_long(cb, d[2], d[3], first, n);
    if (looked) return;
    looked = true;
    if (all12()) return;
    drop_long();
    ok = alloc_long(18);
    if (ok) put_long(cb, d[2], d[3], first, n);
  });
  if (!ok) return done(false);
  if (L->recon == 12 && !all12()) {
    drop_long();
    if (!alloc_long(18)) return done(false);
    host_to_device(a + 2, 2, vh, rh.n, stage, [&](char *const *d, size_t site, size_t n) {
      put_long(rh.parity(site), d[0], d[1], rh.local(site), n);
    });
  }
  return done(true);
}

template <typename T>
static void extract_L(T *fat, T *lng, const typename Handles<T>::L *L, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:extract_L");
  QPHIX_REQUIRE(L && fat && lng, "extract_L: null argument");
  const int vh = ctx().g.vh;
  const RawHalves rh(evenodd & ((L->fat[0] ? QPHIX_EVEN : 0) | (L->fat[1] ? QPHIX_ODD : 0)));
  char *stage = (char *)dev_alloc(host_stage_bytes(2 * 72 * sizeof(T), vh, std::max(rh.n, 1)));
  if (!stage) return;  // error recorded
  const HostArray a[2] = {rh.array(fat, 72), rh.array(lng, 72)};
  device_to_host(a, 2, vh, rh.n, stage, [&](char *const *d, size_t first, size_t n) {
    const int cb = rh.parity(first);
    hipLaunchKernelGGL(k_export_fwd<T>, dim3((unsigned)(n / 64), 2), dim3(256), 0, ctx().stream, L->fat[cb],
                       L->lng[cb], L->lsign[cb], rh.local(first), L->recon == 12 ? 6 : 9, (T *)d[0], (T *)d[1]);
    HIP_CHECK(hipGetLastError());
  });
  dev_free(stage);
}

template <typename T> static void destroy_L(typename Handles<T>::L *L) {
  if (!L) return;
  if (ctx().initialised) HIP_CHECK(hipStreamSynchronize(ctx().stream));
  links_free<T>(L);
  delete L;
}

template <typename T> static void backcheck(const LinksT<T> *L, double out[4]) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:backcheck");
  QPHIX_REQUIRE(L && L->fat[0] && L->fat[1], "backcheck needs both parities");
  const Geometry &gg = ctx().g;
  Geo g{gg.nxh, gg.ny, gg.nz, gg.nt, gg.vh, gg.nxy, gg.nxyz};
  unsigned long long *d = (unsigned long long *)dev_alloc(sizeof(unsigned long long) * 4);
  if (!d) return;  // error recorded
  HIP_CHECK(hipMemsetAsync(d, 0, sizeof(unsigned long long) * 4, ctx().stream));
  const int ncl = L->recon == 12 ? 6 : 9;
  for (int cb = 0; cb < 2; ++cb)
    hipLaunchKernelGGL(k_backcheck<T>, dim3(nblk(gg.vh)), dim3(256), 0, ctx().stream, L->fat[cb],
                       L->lng[cb], L->lsign[cb], L->fat[1 - cb], L->lng[1 - cb], L->lsign[1 - cb],
                       ncl, g, cb, d);
  unsigned long long h[4];
  d2h(h, d, sizeof(h));
  sync();
  for (int k = 0; k < 4; ++k) std::memcpy(&out[k], &h[k], sizeof(double));
  dev_free(d);
}

// Raw gauge links ([i][mu][3][3][re,im]) of the sites [first, first + n) of one
// parity <-> complex-major layout.
template <typename T>
__global__ void __launch_bounds__(256) k_gauge_in(T *dst, const T *raw, int vh, int first) {
  __shared__ __align__(16) T tile[RAW_TILE_REALS];
  const int base = blockIdx.x * 64, lane = threadIdx.x & 63;
  raw_tile_in<T>(tile, raw + 72 * (size_t)base);
  const cplx<T> *mine = reinterpret_cast<const cplx<T> *>(tile + RAW_TILE_STRIDE * lane);
  cplx<T> *d = reinterpret_cast<cplx<T> *>(dst) + first + base + lane;
  for (int q = threadIdx.x >> 6; q < 36; q += 4) d[(size_t)q * (size_t)vh] = mine[q];
}

template <typename T>
__global__ void __launch_bounds__(256) k_gauge_out(T *raw, const T *src, int vh, int first) {
  __shared__ __align__(16) T tile[RAW_TILE_REALS];
  const int base = blockIdx.x * 64, lane = threadIdx.x & 63;
  cplx<T> *mine = reinterpret_cast<cplx<T> *>(tile + RAW_TILE_STRIDE * lane);
  const cplx<T> *s = reinterpret_cast<const cplx<T> *>(src) + first + base + lane;
  for (int q = threadIdx.x >> 6; q < 36; q += 4) mine[q] = s[(size_t)q * (size_t)vh];
  raw_tile_out<T>(raw + 72 * (size_t)base, tile);
}

// Per link of one parity (complex-major): |r2 - conj(r0 x r1)|, the largest
// over the links into *maxbits (as the bits of a non-negative double).
template <typename T> __global__ void k_gauge_su3_check(const T *u, int vh, unsigned long long *maxbits) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double worst = 0;
  if (i < vh) {
    for (int mu = 0; mu < 4; ++mu) {
      double re[9], im[9];
      for (int e = 0; e < 9; ++e) {
        re[e] = u[2 * gauge_elem(mu, e, i, vh)];
        im[e] = u[2 * gauge_elem(mu, e, i, vh) + 1];
      }
      for (int c = 0; c < 3; ++c) {
        const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
        const double xr = re[c1] * re[3 + c2] - im[c1] * im[3 + c2] - (re[c2] * re[3 + c1] - im[c2] * im[3 + c1]);
        const double xi = re[c1] * im[3 + c2] + im[c1] * re[3 + c2] - (re[c2] * im[3 + c1] + im[c2] * re[3 + c1]);
        worst = fmax(worst, fabs(re[6 + c] - xr));
        worst = fmax(worst, fabs(im[6 + c] + xi));
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) worst = fmax(worst, __shfl_down(worst, off, 64));
  if ((threadIdx.x & 63) == 0) atomic_max_nonneg(maxbits, worst);
}

// Rows 0-1 of every link, complex-major with 6 elements per link.
template <typename T> __global__ void k_gauge_rows(T *dst, const T *u, int vh) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  for (int mu = 0; mu < 4; ++mu)
    for (int e = 0; e < 6; ++e) {
      dst[2 * gauge_elem_n(mu, e, i, vh, 6)] = u[2 * gauge_elem(mu, e, i, vh)];
      dst[2 * gauge_elem_n(mu, e, i, vh, 6) + 1] = u[2 * gauge_elem(mu, e, i, vh) + 1];
    }
}

static int g_gauge_recon_mode = 0;  // 18: never keep the two-row copy

// ------------------------------------------------------------------ G, F
// Gauge field: all links are always loaded (the reference reads both raw
// blocks whatever the parity, qphix_d3.cpp:198-200); EVENODD is recorded as
// EVEN (qphix_d3.cpp:195).
template <typename T> static typename Handles<T>::G *create_G(const T *raw, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:create_G", nullptr);
  QPHIX_REQUIRE(raw, "create_G: null array", nullptr);
  QPHIX_REQUIRE(evenodd == QPHIX_EVENODD || evenodd == QPHIX_EVEN || evenodd == QPHIX_ODD,
                "create_G: bad parity", nullptr);
  const int vh = ctx().g.vh;
  const size_t n = 72 * (size_t)vh;
  char *stage = (char *)dev_alloc(host_stage_bytes(72 * sizeof(T), vh, 2));
  if (!stage) return nullptr;
  auto *G = new typename Handles<T>::G;
  G->parity = evenodd == QPHIX_EVENODD ? QPHIX_EVEN : evenodd;
  for (int cb = 0; cb < 2; ++cb) {
    G->u[cb] = (T *)dev_alloc(sizeof(T) * n);
    if (!G->u[cb]) {  // error recorded
      sync();
      dev_free(G->u[0]);
      dev_free(stage);
      delete G;
      return nullptr;
    }
  }
  const RawHalves rh(QPHIX_EVENODD);
  const HostArray a = rh.array(raw, 72);
  host_to_device(&a, 1, vh, 2, stage, [&](char *const *d, size_t first, size_t m) {
    hipLaunchKernelGGL(k_gauge_in<T>, dim3((unsigned)(m / 64)), dim3(256), 0, ctx().stream, G->u[rh.parity(first)],
                       (const T *)d[0], vh, rh.local(first));
    HIP_CHECK(hipGetLastError());
  });
  dev_free(stage);
  // Two-row copy for the force kernel when every link is SU(3) to rounding
  // (the exact links stay in u for extract_G).
  bool su3 = g_gauge_recon_mode != 18;
  unsigned long long *dmax = su3 ? (unsigned long long *)dev_try_alloc(sizeof(unsigned long long)) : nullptr;
  if (!dmax) su3 = false;
  if (su3) {
    HIP_CHECK(hipMemsetAsync(dmax, 0, sizeof(unsigned long long), ctx().stream));
    for (int cb = 0; cb < 2; ++cb)
      hipLaunchKernelGGL(k_gauge_su3_check<T>, dim3(nblk(vh)), dim3(256), 0, ctx().stream, G->u[cb], vh, dmax);
    HIP_CHECK(hipGetLastError());
    unsigned long long bits = 0;
    d2h(&bits, dmax, sizeof(bits));
    sync();
    double worst;
    std::memcpy(&worst, &bits, sizeof(worst));
    su3 = worst <= recon_tol<T>();
  }
  dev_free(dmax);
  if (su3) {
    for (int cb = 0; cb < 2; ++cb) G->u12[cb] = (T *)dev_try_alloc(sizeof(T) * 48 * (size_t)vh);
    if (!G->u12[0] || !G->u12[1]) {  // no room: the force kernel reads the full links
      dev_free(G->u12[0]);
      dev_free(G->u12[1]);
      G->u12[0] = G->u12[1] = nullptr;
    } else {
      for (int cb = 0; cb < 2; ++cb) {
        hipLaunchKernelGGL(k_gauge_rows<T>, dim3(nblk(vh)), dim3(256), 0, ctx().stream, G->u12[cb],
                           G->u[cb], vh);
        HIP_CHECK(hipGetLastError());
      }
    }
  }
  sync();
  return G;
}

template <typename T> static void extract_G(T *raw, const typename Handles<T>::G *G, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:extract_G");
  QPHIX_REQUIRE(raw && G, "extract_G: null argument");
  const int vh = ctx().g.vh;
  const RawHalves rh(evenodd);
  char *stage = (char *)dev_alloc(host_stage_bytes(72 * sizeof(T), vh, std::max(rh.n, 1)));
  if (!stage) return;
  const HostArray a = rh.array(raw, 72);
  device_to_host(&a, 1, vh, rh.n, stage, [&](char *const *d, size_t first, size_t m) {
    hipLaunchKernelGGL(k_gauge_out<T>, dim3((unsigned)(m / 64)), dim3(256), 0, ctx().stream, (T *)d[0],
                       G->u[rh.parity(first)], vh, rh.local(first));
    HIP_CHECK(hipGetLastError());
  });
  dev_free(stage);
}

template <typename T> static void destroy_G(typename Handles<T>::G *G) {
  if (!G) return;
  if (ctx().initialised) HIP_CHECK(hipStreamSynchronize(ctx().stream));
  dev_free(G->u[0]);
  dev_free(G->u[1]);
  dev_free(G->u12[0]);
  dev_free(G->u12[1]);
  delete G;
}

// Momentum: both parities are always held (zero unless loaded), the requested
// parities are loaded (qphix_d3.cpp:360-488).
template <typename T> static typename Handles<T>::F *create_F(const T *raw, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:create_F", nullptr);
  QPHIX_REQUIRE(raw, "create_F: null array", nullptr);
  QPHIX_REQUIRE(evenodd == QPHIX_EVENODD || evenodd == QPHIX_EVEN || evenodd == QPHIX_ODD,
                "create_F: bad parity", nullptr);
  const int vh = ctx().g.vh;
  const RawHalves rh(evenodd);
  char *stage = (char *)dev_alloc(host_stage_bytes(72 * sizeof(T), vh, rh.n));
  if (!stage) return nullptr;  // error recorded
  auto *F = new typename Handles<T>::F;
  F->parity = evenodd == QPHIX_EVENODD ? QPHIX_EVEN : evenodd;
  for (int cb = 0; cb < 2; ++cb) {
    F->h[cb] = (T *)dev_alloc(sizeof(T) * 32 * (size_t)vh);
    if (!F->h[cb]) {  // error recorded
      sync();
      dev_free(F->h[0]);
      dev_free(stage);
      delete F;
      return nullptr;
    }
    if (!(evenodd & (cb ? QPHIX_ODD : QPHIX_EVEN)))
      HIP_CHECK(hipMemsetAsync(F->h[cb], 0, sizeof(T) * 32 * (size_t)vh, ctx().stream));
  }
  const HostArray a = rh.array(raw, 72);
  host_to_device(&a, 1, vh, rh.n, stage, [&](char *const *d, size_t first, size_t m) {
    hipLaunchKernelGGL(k_mom_in<T>, dim3(nblk(4 * (int)m)), dim3(256), 0, ctx().stream,
                       F->h[rh.parity(first)] + 32 * (size_t)rh.local(first), (const T *)d[0], 4 * (int)m);
    HIP_CHECK(hipGetLastError());
  });
  dev_free(stage);
  return F;
}

template <typename T> static void extract_F(T *raw, const typename Handles<T>::F *F, int evenodd) {
  QPHIX_REQUIRE(require_init(), "QPHIX_init has not been called:extract_F");
  QPHIX_REQUIRE(raw && F, "extract_F: null argument");
  const int vh = ctx().g.vh;
  const RawHalves rh(evenodd);
  char *stage = (char *)dev_alloc(host_stage_bytes(72 * sizeof(T), vh, std::max(rh.n, 1)));
  if (!stage) return;  // error recorded
  const HostArray a = rh.array(raw, 72);
  device_to_host(&a, 1, vh, rh.n, stage, [&](char *const *d, size_t first, size_t m) {
    hipLaunchKernelGGL(k_mom_out<T>, dim3(nblk(4 * (int)m)), dim3(256), 0, ctx().stream, (T *)d[0],
                       F->h[rh.parity(first)] + 32 * (size_t)rh.local(first), 4 * (int)m);
    HIP_CHECK(hipGetLastError());
  });
  dev_free(stage);
}

template <typename T> static void destroy_F(typename Handles<T>::F *F) {
  if (!F) return;
  if (ctx().initialised) HIP_CHECK(hipStreamSynchronize(ctx().stream));
  dev_free(F->h[0]);
  dev_free(F->h[1]);
  delete F;
}

} // namespace qphix

using namespace qphix;

extern "C" {

#define QPHIX_FIELD_API(P, T)                                                                     \
  QPHIX_##P##3_ColorVector *QPHIX_##P##3_create_V_from_raw(T *src, QPHIX_evenodd_t evenodd) {     \
    return create_V<T>(src, evenodd);                                                             \
  }                                                                                               \
  void QPHIX_##P##3_extract_V_to_raw(T *dest, QPHIX_##P##3_ColorVector *src, QPHIX_evenodd_t) {   \
    extract_V<T>(dest, src);                                                                      \
  }                                                                                               \
  void QPHIX_##P##3_destroy_V(QPHIX_##P##3_ColorVector *V) { destroy_V<T>(V); }                   \
  QPHIX_##P##3_FermionLinksAsqtad *QPHIX_##P##3_asqtad_create_L_from_raw(                         \
      T *fat, T *lng, T *fatback, T *lngback, QPHIX_evenodd_t evenodd) {                          \
    return create_L<T>(fat, lng, fatback, lngback, evenodd);                                      \
  }                                                                                               \
  void QPHIX_##P##3_asqtad_extract_L_to_raw(T *fat, T *lng, QPHIX_##P##3_FermionLinksAsqtad *src, \
                                            QPHIX_evenodd_t evenodd) {                            \
    extract_L<T>(fat, lng, src, evenodd);                                                         \
  }                                                                                               \
  void QPHIX_##P##3_asqtad_destroy_L(QPHIX_##P##3_FermionLinksAsqtad *L) { destroy_L<T>(L); }    \
  int QPHIX_##P##3_asqtad_links_recon(QPHIX_##P##3_FermionLinksAsqtad *L) {                       \
    return L ? L->recon : 0;                                                                      \
  }                                                                                               \
  QPHIX_##P##3_GaugeField *QPHIX_##P##3_create_G_from_raw(T *raw, QPHIX_evenodd_t evenodd) {      \
    return create_G<T>(raw, evenodd);                                                             \
  }                                                                                               \
  void QPHIX_##P##3_extract_G_to_raw(T *raw, QPHIX_##P##3_GaugeField *G, QPHIX_evenodd_t eo) {    \
    extract_G<T>(raw, G, eo);                                                                     \
  }                                                                                               \
  void QPHIX_##P##3_destroy_G(QPHIX_##P##3_GaugeField *G) { destroy_G<T>(G); }                    \
  int QPHIX_##P##3_gauge_links_recon(QPHIX_##P##3_GaugeField *G) {                                \
    return G && G->u12[0] ? 12 : 18;                                                              \
  }                                                                                               \
  QPHIX_##P##3_Force *QPHIX_##P##3_create_F_from_raw(T *raw, QPHIX_evenodd_t evenodd) {           \
    return create_F<T>(raw, evenodd);                                                             \
  }                                                                                               \
  void QPHIX_##P##3_extract_F_to_raw(T *raw, QPHIX_##P##3_Force *F, QPHIX_evenodd_t eo) {         \
    extract_F<T>(raw, F, eo);                                                                     \
  }                                                                                               \
  void QPHIX_##P##3_destroy_F(QPHIX_##P##3_Force *F) { destroy_F<T>(F); }

QPHIX_FIELD_API(D, double)
QPHIX_FIELD_API(F, float)

void QPHIX_MI355X_set_long_recon(int mode) { g_recon_mode = mode == 18 ? 18 : 0; }
void QPHIX_MI355X_set_gauge_recon(int mode) { g_gauge_recon_mode = mode == 18 ? 18 : 0; }
void QPHIX_MI355X_set_sloppy_link_bits(int bits) { g_sloppy_link_bits = bits == 16 ? 16 : 32; }
void QPHIX_MI355X_set_sloppy_long_recon(int recon) { g_sloppy_long_recon = recon == 12 ? 12 : 8; }

void QPHIX_D3_asqtad_links_backcheck(QPHIX_D3_FermionLinksAsqtad *L, double out[4]) {
  backcheck<double>(L, out);
}

} // extern "C"
