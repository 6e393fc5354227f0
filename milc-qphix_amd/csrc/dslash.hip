// dslash.hip -- even-odd asqtad/HISQ Dslash for gfx950.
//
// Replaces the reference's per-parity site loop (ks_long_dslash.cpp:564-668)
// and its absent codegen kernel body (ks_dslash_complete_specialization.cpp:14-54):
//   out(x) = sum_mu [ F_{2mu+1}(x) in(x+mu) + F_{2mu}(x) in(x-mu)
//                   + N_{2mu+1}(x) in(x+3mu) + N_{2mu}(x) in(x-3mu) ]
// for every site x of the output parity, with the 16 links applied as stored
// (1146 flops/site).  One work-item per output site; neighbour indices come from
// coordinate arithmetic with periodic wrap (no neighbour table, no halo: the
// reference's boundary.cpp / ks_boundary face exchange has no counterpart on one
// GPU).  Links stream from HBM once per application in 16-byte coalesced
// chunks; the 16 neighbour spinor reads per site hit L2 / Infinity Cache.
//
// Fused epilogues remove whole vector passes from the solvers:
//   EPI_PKP     out = D in + s*p, reduce p.out      (calc_pkp, ks_d_congrad_fn.cpp:159-171)
//   EPI_RESTART r = b + D in + s*x, p = r, reduce |r|^2 and the relative residue
//                                                   (calc_rsq, ks_d_congrad_fn.cpp:82-99;
//                                                    relative_residue, ks_blas_utils_c.cpp:110-149)
//   EPI_PKP_FS  out = D in + s*p, reduce p.out, r.out, out.out and r.r: the one
//               reduction of a single-reduction (FEWSUMS) CG step
//                                                   (ks_d_congrad_fn.cpp:150-158, 450-541)
#include "blas.h"
#include "dslash_kernel.h"

namespace qphix {

// Kernel variants of the launches (see dslash_kernel.h).
//
// Links that do not fit the 256 MB Infinity Cache with those of the other
// parity (a solver's next application) are streamed, and so is the output:
// measured at 32^4 (Naik 12, tile-major links), XCD slabs + streaming link
// loads take FP64 from 230 to 201 us and FP32 from 104 to 95 us; streaming
// output stores take them to 188 and 93 us.  The output stores stream even
// where the next kernel reads the result (a solver's tmp = D p): that pair of
// Dslashes is 3% faster than with cached stores (FP32 190 vs 196 us, FP64 390
// vs 403 us).
// Links that do fit are loaded and stored through the caches: the two
// applications of a CG step then take (us each, streamed / cached) FP64
// 12^3x20 18.1 / 12.6, 16^4 19.9 / 14.1, 16^3x32 (252 MB) 24.5 / 22.0, but with
// 18-real Naik links (302 MB) 27.1 / 27.6 and at 20^3x24 (369 MB) 36.2 / 37.4;
// FP32 16^4 10.4 / 7.9, 20^3x24 (184 MB) 19.9 / 16.0, 24^4 (319 MB) 31.7 / 31.7;
// the mixed solver's step with 8-real links (276 MB at 24^4) 74.1 / 69.6.
constexpr int OPT_STREAMED = OPT_XCD | OPT_NTL | OPT_NTS;
constexpr int OPT_CACHED = OPT_XCD;
constexpr size_t LINKS_CACHED = (size_t)272 << 20;  // link bytes of both parities

// Blocks of one wavefront leave no part-filled last round of blocks (FP64 pair,
// us each, 256 / 64 work-items: 24^4 58.1 / 57.2, 24^3x48 116.1 / 111.1).  From
// SMALL_BLOCKS sites on they leave so many partial sums that the vector kernels
// that add them lose more (FP64 CG step at 24^3x48 271.7 / 260.6, at 32^4 400 /
// 404).
constexpr int SMALL_BLOCKS = 400000;

// Under QUAD_SITES sites per parity four lanes share a site (k_dslash_quad), in
// blocks of one wavefront under QUAD_SMALL sites.  A CG step, one lane per site
// / four, blocks of 64 / of 256: FP64 8^4 24.0 / 17.1 / 18.5 us, 12^4 33.9 / 23.5
// / 22.8, 12^3x20 36.0 / 26.8 / 28.6 (18-real Naik 35.9 / 30.1 / 32.4), 16^4 40.6
// / 36.8 / 36.0 (40.9 / 41.5 / 40.9), 16^3x24 47.8 / 48.6 / 45.9 (51.5 / 55.0 /
// 52.7); mixed 8^4 19.1 / 14.3 / 15.8, 16^4 26.1 / 26.5 / 24.3, 16^3x24 29.6 /
// 30.4 / 29.3.
constexpr int QUAD_SMALL = 20000, QUAD_SITES = 40000;
bool dslash_quad(int vh) { return vh < QUAD_SITES; }
// a partial sum per 16 sites under QUAD_SMALL must fit Context::max_blocks
// (vh / 64 + 1024), and links there are always cached
static_assert(QUAD_SMALL / 16 <= QUAD_SMALL / 64 + 1024, "partials of k_dslash_quad");
static_assert((size_t)QUAD_SITES * 2 * 4 * 16 * 36 <= LINKS_CACHED, "k_dslash_quad loads through the caches");

// (Measured and dropped: each XCD walking a z-region t-slice by t-slice
// instead of a t-slab, as the multi-RHS kernels do -- FP64 169.5 vs 170.0 us,
// FP32 87.7 vs 87.3 us at 32^4: one source's +-3 t-slice window already fits.
// Four or eight wavefronts per 64 sites, one per direction or link pair, their
// sums meeting in LDS: 17.8 -> 19.2 us at 12^3x20, 168 -> 186 at 32^4.  Eight
// lanes a site, forward and back links apart, FP64: a CG step 17.0 -> 15.8 us at
// 8^4, but 22.7 / 22.6 at 12^4 and 26.0 / 27.7 at 12^3x20.)
template <typename TL, int NL, typename SI, typename SO, int EPI>
static int launch_one(const DslashKArgs<TL, SI, SO> &a) {
  const int vh = a.g.vh;
  if (dslash_quad(vh)) {
    const int block = vh < QUAD_SMALL ? 64 : 256, nb = vh / (block / 4);
    hipLaunchKernelGGL((k_dslash_quad<TL, NL, SI, SO, EPI, OPT_CACHED>), dim3(nb), dim3(block), 0, ctx().stream, a);
    return nb;
  }
  const size_t links = (size_t)2 * vh * 4 * 16 * (link_nch<TL>(18) + link_nch<TL>(NL));
  const int block = vh < SMALL_BLOCKS ? 64 : DSLASH_BLOCK;
  const int nb = (vh + block - 1) / block;
  if (links <= LINKS_CACHED)
    hipLaunchKernelGGL((k_dslash<TL, NL, SI, SO, EPI, OPT_CACHED>), dim3(nb), dim3(block), 0, ctx().stream, a);
  else
    hipLaunchKernelGGL((k_dslash<TL, NL, SI, SO, EPI, OPT_STREAMED>), dim3(nb), dim3(block), 0, ctx().stream, a);
  return nb;
}

template <typename TL, int NL, typename SI, typename SO>
static int launch_epi(const DslashKArgs<TL, SI, SO> &a, int epi) {
  if (epi == EPI_PLAIN) return launch_one<TL, NL, SI, SO, EPI_PLAIN>(a);
  if (epi == EPI_PKP) return launch_one<TL, NL, SI, SO, EPI_PKP>(a);
  if (epi == EPI_PKP_FS) return launch_one<TL, NL, SI, SO, EPI_PKP_FS>(a);
  return launch_one<TL, NL, SI, SO, EPI_RESTART>(a);
}

template <typename TL, typename SI, typename SO>
static int dispatch(const DslashKArgs<TL, SI, SO> &a, int recon, int epi) {
  int nb = 0;
  if (recon == 8) {  // built for the FP32 sloppy operator only
    if constexpr (std::is_same<TL, float>::value) nb = launch_epi<TL, 8, SI, SO>(a, epi);
    else QPHIX_REQUIRE(false, "Dslash: 8-real long links are FP32 only", 0);
  } else if (recon == 12) {
    nb = launch_epi<TL, 12, SI, SO>(a, epi);
  } else {
    nb = launch_epi<TL, 18, SI, SO>(a, epi);
  }
  HIP_CHECK(hipGetLastError());
  // a step's sums are left to the kernels that need them
  if (epi == EPI_RESTART) reduce_finish(2, nb, a.rc, a.gate);
  return nb;
}

static Geo make_geo() {
  const Geometry &g = ctx().g;
  return Geo{g.nxh, g.ny, g.nz, g.nt, g.vh, g.nxy, g.nxyz};
}

template <typename TL, typename SI, typename SO>
static DslashKArgs<TL, SI, SO> make_args(const LinksT<TL> &L, int cb, SO *out, const SI *in,
                                         const DslashExtra &ex) {
  DslashKArgs<TL, SI, SO> a{};
  a.fat = reinterpret_cast<const typename vec16<TL>::type *>(L.fat[cb]);
  a.lng = reinterpret_cast<const typename vec16<TL>::type *>(L.lng[cb]);
  a.lsign = L.lsign[cb];
  a.in = in;
  a.out = out;
  a.g = make_geo();
  a.cb = cb;
  a.s = (typename link_compute<TL>::type)ex.s;
  a.aux = reinterpret_cast<const SI *>(ex.aux);
  a.b = reinterpret_cast<const SI *>(ex.b);
  a.r = reinterpret_cast<SO *>(ex.r);
  a.p = reinterpret_cast<SO *>(ex.p);
  a.rc = reduce_ctl(reinterpret_cast<SolverState *>(ex.state), ex.scalar_op);
  a.gate = ex.gate;
  return a;
}

template <typename T>
int launch_dslash(const LinksT<T> &L, int cb, T *out, const T *in, int epi, const DslashExtra &ex) {
  QPHIX_REQUIRE(L.fat[cb] && L.lng[cb] && in && out, "Dslash: links or vectors of this parity missing", 0);
  return dispatch<T, T, T>(make_args<T, T, T>(L, cb, out, in, ex), L.recon, epi);
}

template int launch_dslash<double>(const LinksT<double> &, int, double *, const double *, int,
                                    const DslashExtra &);
template int launch_dslash<float>(const LinksT<float> &, int, float *, const float *, int,
                                   const DslashExtra &);

// FP16-stored spinors with FP32 links and arithmetic.  out_h (half) or
// out_f (float) receives the result.
int launch_dslash_half(const LinksT<float> &L, int cb, HalfSite *out_h, float *out_f,
                        const HalfSite *in, int epi, const DslashExtra &ex) {
  QPHIX_REQUIRE(L.fat[cb] && L.lng[cb] && in && (out_h || out_f), "Dslash: links or vectors of this parity missing", 0);
  if (out_h)
    return dispatch<float, HalfSite, HalfSite>(make_args<float, HalfSite, HalfSite>(L, cb, out_h, in, ex), L.recon, epi);
  return dispatch<float, HalfSite, float>(make_args<float, HalfSite, float>(L, cb, out_f, in, ex), L.recon, epi);
}

int launch_dslash_q16(const LinksT<Q16> &L, int cb, float *out, const float *in, int epi,
                       const DslashExtra &ex) {
  QPHIX_REQUIRE(L.fat[cb] && L.lng[cb] && in && out, "Dslash: links or vectors of this parity missing", 0);
  return dispatch<Q16, float, float>(make_args<Q16, float, float>(L, cb, out, in, ex), L.recon, epi);
}

int launch_dslash_q16_half(const LinksT<Q16> &L, int cb, HalfSite *out_h, float *out_f, const HalfSite *in,
                            int epi, const DslashExtra &ex) {
  QPHIX_REQUIRE(L.fat[cb] && L.lng[cb] && in && (out_h || out_f), "Dslash: links or vectors of this parity missing", 0);
  if (out_h)
    return dispatch<Q16, HalfSite, HalfSite>(make_args<Q16, HalfSite, HalfSite>(L, cb, out_h, in, ex), L.recon, epi);
  return dispatch<Q16, HalfSite, float>(make_args<Q16, HalfSite, float>(L, cb, out_f, in, ex), L.recon, epi);
}

} // namespace qphix
