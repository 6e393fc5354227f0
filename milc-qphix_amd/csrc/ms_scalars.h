// ms_scalars.h -- the scalar recurrences of the multi-shift solvers, one shift
// per work-item of one block per source (MAXNDMASS <= MS_BLOCK).
//
// Serial in one thread the recurrences of a step were a chain of dependent state
// reads, divisions and writes per shift (k_finalize 5.7 us at 9 shifts, the
// batched solver's 16 us at 7); here every shift's state is in registers, read
// once.  The arithmetic per shift is the reference's (ks_multicg_offset.cpp:463-598).
#pragma once
#include "reduce.h"

namespace qphix {

constexpr int MS_BLOCK = 256;
static_assert(MAXNDMASS <= MS_BLOCK, "one work-item per shift");

// Shift threadIdx.x of the state: zeta_i, zeta_{i-1}, zeta_{i+1}, beta_i, alpha.
struct MsShift {
  double zi, zim1, zip1, bi, al;
  int fin;
};
__device__ __forceinline__ MsShift ms_load(const SolverState *s, int j) {
  return MsShift{s->zeta_i[j], s->zeta_im1[j], s->zeta_ip1[j], s->beta_i[j], s->alpha[j], s->finished[j]};
}

// End of the previous step, before its coefficients are overwritten: kept for
// the shifted systems' next update when theirs waits (s->defer), else nothing is
// pending any more; shifts that took their last update retire.  Every work-item
// of the block calls it.
__device__ __forceinline__ void ms_commit(SolverState *s, int j, const MsShift &x) {
  const int q = s->pend, n = s->num_now;
  const bool wait = s->defer != 0;
  if (j < n) {
    if (wait) {
      s->pbeta[q][j] = x.bi;
      s->palpha[q][j] = x.al;
      s->pzeta[q][j] = x.zip1;
    }
    if (s->sdone[j] == 2) s->sdone[j] = 1;
  }
  __syncthreads();
  if (j == 0) {
    if (wait) s->pend_nn[q] = n;
    s->pend = wait ? q + 1 : 0;
    s->defer = 0;
    s->open = 0;
  }
  __syncthreads();
}

// zeta_{i+1} and beta_i from the base system's beta bl (:463-496); bim1 and al
// its previous beta and alpha.  R: the solver's type.
template <typename R>
__device__ __forceinline__ void ms_zeta_beta(MsShift &x, double shift, bool low, double bl_, double bim1_, double al_) {
  if (low) {
    x.bi = bl_;
    x.zip1 = 1.0;
    return;
  }
  const R zi = (R)x.zi, zim1 = (R)x.zim1, bim1 = (R)bim1_, bl = (R)bl_, al = (R)al_, sh = (R)shift;
  R zip1 = zi * zim1 * bim1;
  const R c1 = bl * al * (zim1 - zi);
  const R c2 = (R)(zim1 * bim1 * (1.0 + sh * bl));
  R bj;
  if (c1 + c2 != (R)0.0) zip1 /= c1 + c2;
  else { zip1 = 0; x.fin = 1; }
  if (zi != (R)0.0) bj = bl * zip1 / zi;
  else { zip1 = 0; bj = 0; x.fin = 1; }
  x.zip1 = zip1;
  x.bi = bj;
}

// alpha from the base system's alpha alow (:504-598).
template <typename R> __device__ __forceinline__ void ms_alpha(MsShift &x, bool low, double bl_, double alow) {
  if (low) {
    x.al = alow;
    return;
  }
  const R zi = (R)x.zi, bl = (R)bl_;
  if (zi * bl != (R)0.0) x.al = (R)alow * (R)x.zip1 * (R)x.bi / (zi * bl);
  else { x.al = 0; x.fin = 1; }
}

// Shifts still advancing after ms_zeta_beta: the last one leaves when it is
// finished (one a step, as in the reference's loop).  The same in every work-item.
__device__ __forceinline__ int ms_num_now(int n, int j, int jl, const MsShift &x) {
  __shared__ int drop;
  if (j == 0) drop = 0;
  __syncthreads();
  if (j == n - 1 && j > jl && x.fin) drop = 1;
  __syncthreads();
  return n - drop;
}

__device__ __forceinline__ void ms_store_next(SolverState *s, int j, const MsShift &x) {
  s->alpha[j] = x.al;
  s->beta_im1[j] = x.bi;
  s->zeta_im1[j] = x.zi;
  s->zeta_i[j] = x.zip1;
}

} // namespace qphix
