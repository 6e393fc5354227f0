// blas.h -- solver vector kernels (blas.hip) and their launchers.
#pragma once
#include "reduce.h"

namespace qphix {

constexpr int BLAS_BLOCK = 256;
// Blocks of the vector kernels that sum the previous kernel's partials
// themselves (consumer-side reductions).  Every block reads all of them (at
// 32^4, 2048 Dslash partials x 4 sums: 64 KB per block), so larger blocks read
// fewer bytes but leave fewer wavefronts resident.  cons_block() threads per
// block: 512, on lattices under CONS_SMALL sites per parity 128, which spread
// over more CUs (QPHIX_CONS_BLOCK = 256, 512 or 1024 in the environment),
// compiled for up to CONS_BLOCK_MAX.  Measured at 32^4 (mixed CG, FP32 /
// FP16-stored vectors): 256 -> 0.190 / 0.180 s, 512 -> 0.187 / 0.179 s; 1024
// made the single-reduction update 36.5 us against 21.5 us (half the
// wavefronts resident).  A CG step, 128 / 512: 8^4 23.9 / 25.0 us, 12^4 33.6 /
// 34.8, 16^4 40.3 / 40.6, 16^3x24 48.8 / 47.5; mixed 8^4 19.2 / 20.4, 16^4 26.0 /
// 26.9, 16^3x24 29.4 / 29.8, 16^3x32 33.2 / 32.9.
constexpr int CONS_SMALL = 40000;
constexpr int CONS_BLOCK_MAX = 1024;
int cons_block();
inline int cons_nb(int vh) { return (vh + cons_block() - 1) / cons_block(); }

ReduceCtl reduce_ctl(SolverState *st, int op);
double *reduce_result_ptr();  // where reductions without a state leave their sums

template <typename T> void blas_norm2(const T *v, SolverState *st, int op);
// One CG step after a p.Ap Dslash (nb_pkp blocks of partials): update x, r and
// |r|^2, then p, each kernel summing the previous one's partials itself (no
// finalize launches).  rel: the relative residue is wanted.
template <typename T>
void blas_cg_step_c(T *x, T *p, T *r, const T *ttt, SolverState *st, int *gate, int nb_pkp, bool rel);
double *partials_b();
// One single-reduction (FEWSUMS) CG step after an EPI_PKP_FS Dslash with
// nb_pkp blocks of partials: x, r and p in one pass (k_cg_step_fs).
template <typename T>
void blas_cg_step_fs(T *x, T *p, T *r, const T *ttt, SolverState *st, int *gate, int nb_pkp);
// st's shifts (device array) and their starting values, after STATE_HEAD bytes.
void blas_ms_start(SolverState *st, const double *shifts);
// Which solvers take single-reduction steps (fewsums_mode(), common.h): bit 0
// the one-precision CG (QPHIX_*3_asqtad_invert, when relresid is off), bit 1
// the sloppy steps of the mixed-precision CG.
// After a p.Ap Dslash (nb_pkp blocks of partials): r, |r|^2 and the step's scalars.
template <typename T> void blas_ms_update_r(T *r, const T *ttt, SolverState *st, int nb_pkp, const int *gate);
template <typename T>
void blas_ms_update_pm(T *const *x, T *const *p, const T *r, int nshift, const SolverState *st,
                       const int *gate);
template <typename T>
void blas_ms_update_dest(T *const *x, T *const *p, int nshift, const SolverState *st);
// update_pm with the shifted systems up to st->fuse steps at a time (rprev:
// fuse - 1 saved residuals); flush = true applies what is still pending.
template <typename T>
void blas_ms_update_pm_def(T *const *x, T *const *p, const T *r, T *rprev, int nshift, SolverState *st,
                           const int *gate, bool flush);
void set_int(int *p, int v);

} // namespace qphix
