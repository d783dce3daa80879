// What the BiCGStab of the nodal solves (pressure_guess.hip) and its
// preconditioners (mg.hip) share.
#pragma once
#include "fvm_internal.h"

// The iteration's scalars, kept on the device.  FVM_S_DONE: converged (or NaN); the
// kernels enqueued behind that iteration return at once, so the host can enqueue
// several iterations between two looks at the residual.
enum { FVM_S_RHO = 0, FVM_S_RHO_OLD, FVM_S_ALPHA, FVM_S_OMEGA, FVM_S_RR, FVM_S_BB, FVM_S_ITS, FVM_S_DONE };

// the relative residual is not above rtol (also true for NaN and for b = 0)
__device__ __forceinline__ bool fvm_bcg_done(double rr, double bb, double rtol) {
  return !(sqrt(rr) / sqrt(bb) > rtol);
}
// After an exact solve (r = 0) rho_old and omega are 0: restart with beta = 0
// instead of forming 0/0, so x stays the solution.
__device__ __forceinline__ double fvm_bcg_beta(int first, double rho, const double *sc) {
  const double rho_old = sc[FVM_S_RHO_OLD], omega = sc[FVM_S_OMEGA];
  return first || rho_old == 0.0 || omega == 0.0 ? 0.0 : (rho / rho_old) * (sc[FVM_S_ALPHA] / omega);
}

// One iteration with the one-level preconditioner: the vectors (p, v read, p_new,
// v_new written), the partial sums (fvm_one_partials of them in each array) and the
// scalars.
#define FVM_ONE_BLOCKS 256
#define FVM_ONE_TILE 32  // points a side of a block's tile
static inline int64_t fvm_one_partials(int NX, int NY) {
  const int64_t tiles = (int64_t)((NX + FVM_ONE_TILE - 1) / FVM_ONE_TILE) * ((NY + FVM_ONE_TILE - 1) / FVM_ONE_TILE);
  return tiles > FVM_ONE_BLOCKS ? tiles : FVM_ONE_BLOCKS;
}
struct FvmBcgOne {
  double *x, *r, *s, *t, *y, *z, *p_new, *v_new;
  const double *rh, *p, *v;
  double *prv, *pts, *ptt, *prho, *prr, *sc;
  int n_r;  // partials in prho and prr
  int first;
  double rtol;
};

// Preconditioner of a 5-point system on NX x NY nodes: y = M b stands for the system
// with every row divided by its diagonal d.  scale: the couplings are not divided
// by d yet.  *out is null where no preconditioner is offered.  It belongs to the
// context and lasts until the next build.
int fvm_precond_build(fvm_ctx *ctx, int NX, int NY, const double *d, const double *e, const double *w, const double *s,
                      const double *n, bool scale, fvm_precond **out);
// The multigrid cycle; a one-level preconditioner comes with its own iteration.
bool fvm_precond_one_level(const fvm_precond *m);
int fvm_precond_apply(fvm_ctx *ctx, const fvm_precond *m, const double *b, double *y, const double *sc);
int fvm_precond_one_iteration(fvm_ctx *ctx, const fvm_precond *m, const FvmBcgOne &O);
