// Whole marker steps in the reference's call order (main_subduction.c:227-463),
// enqueued without host round trips except where a scalar must come back.
#include "fvm_internal.h"

extern "C" int fvm_step_thermal(fvm_ctx *ctx, const fvm_grid *g, fvm_markers *mk, const NodalArrays *nf,
                                const Materials *mat, const Options *opt, const BoundaryValues *bv, double dt,
                                int32_t nproj, const fvm_projection *list) {
  if (!ctx || !mk || !nf || !mat || !opt || !bv) return FVM_ERR_ARG;
  FVM_TRY(fvm_grid_check(ctx, g));
  FVM_TRY(fvm_locate_async(ctx, g, mk, 0, mat, true));         // :243 + density :255-264
  if (list)                                                     // :268
    FVM_TRY(fvm_project_marker_fields(ctx, g, mk, nproj, list));
  else
    FVM_TRY(fvm_project_markers_nodes_all2(ctx, g, mk, nf, mat));
  if (!nf->thisT || !nf->lastT || !nf->rho || !nf->Cp || !nf->kThermal || !nf->vx || !nf->vy || !nf->wxy)
    return fvm_set_err(ctx, FVM_ERR_ARG, "step: missing nodal field");
  double *dTsub = nullptr, *deltaT = nullptr;                   // :415 subgridTemperatureChanges
  // marker T is unchanged since the projection above, so its bucket-ordered
  // copy can be reused by the fused dTsub pass
  ctx->reuse_payload = true;
  const int rc = fvm_subgrid_t_pass1(ctx, nf->thisT, g, nf, mk, mat, dt, opt->subgridTemperatureDiffusivity, &dTsub,
                                     &deltaT);
  ctx->reuse_payload = false;
  FVM_TRY(rc);
  // its pass 2 runs inside the advection kernel (:435 advectMarkersRK)
  FVM_TRY(fvm_advect_with_subgrid_t2(ctx, mk, nf, g, bv, dt, deltaT, dTsub, dt));
  return FVM_OK;
}

// The part of a visco-elasto-plastic step behind the Stokes solve, for complete
// arguments: the calls of fvm_step_vep's plain path in fewer passes over the
// markers, which are what bounds a large step (12.6 us for each 64-bit column of
// 8 M markers).
//   - subgrid T pass 1 right behind the projection, while its bucket-ordered T
//     is still there (it writes workspace only, so an error below leaves T alone);
//   - the subgrid stress changes formed in the strain pass, whose gathers they
//     share, and kept apart from the stresses until the residual has been found
//     to be a number;
//   - one wait for that flag and for the residual;
//   - the changes, the stress update and the rotation behind each marker's
//     advection, with subgrid T pass 2 in front of it.
// Every value is formed by the same operations in the same order as there.
// 801 x 401 nodes, 8 M markers: strain + subgrid stress + stress update + subgrid T2
// + RK4 + rotation took 222 + 166 + 125 + 74 + 353 + 150 us in passes of their own.
static int vep_after_stokes(fvm_ctx *ctx, const fvm_grid *g, fvm_markers *mk, const NodalArrays *nf,
                            const NodalArrays *host, const Materials *mat, const Options *opt,
                            const BoundaryValues *bv, double dt, double *residual) {
  const size_t cs = ((size_t)mk->nMark + 31) / 32 * 32, nn = ((size_t)g->NX * g->NY + 31) / 32 * 32;
  const bool sub = opt->subgridStressDiffusivity > 0.0;
  FVM_TRY(fvm_ws(ctx, ctx->scratch, (cs * (sub ? 4 : 1) + 2 * nn) * sizeof(double)));
  double *deltaT = (double *)ctx->scratch.ptr, *srr = deltaT + nn, *dTsub = srr + nn;
  double *dxx = sub ? dTsub + cs : nullptr, *dyy = sub ? dxx + cs : nullptr, *dxy = sub ? dyy + cs : nullptr;
  ctx->reuse_payload = true;  // T is as it was projected
  const int rc = fvm_subgrid_t_into(ctx, host->thisT, g, nf, mk, mat, dt, opt->subgridTemperatureDiffusivity, dTsub,
                                    deltaT);
  ctx->reuse_payload = false;
  FVM_TRY(rc);
  int32_t *bad = (int32_t *)ctx->pinned.ptr;
  double *sum = (double *)ctx->pinned.ptr + 8;
  *bad = 0;
  FVM_TRY(fvm_launch_strain_pressure(ctx, g, host, mk, dt, bad, opt->subgridStressDiffusivity, dxx, dyy, dxy));
  FVM_TRY(fvm_enqueue_strain_rate_residual(ctx, g, mk, srr, sum));
  FVM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (*bad) return fvm_set_err(ctx, FVM_ERR_NAN_RESIDUAL, "NaN strain rate residual on an active marker");
  if (sub) FVM_TRY(fvm_project_stress_changes(ctx, g, host, mk, dxx, dyy, dxy));
  FVM_TRY(fvm_advect_with_stress(ctx, mk, host, g, bv, dt, deltaT, dTsub, dxx, dyy, dxy));
  if (residual) *residual = *sum / (g->LX * g->LY);
  return FVM_OK;
}

extern "C" int fvm_step_vep(fvm_ctx *ctx, const fvm_grid *g, fvm_markers *mk, const NodalArrays *nf,
                            const NodalArrays *host, const Materials *mat, const Options *opt,
                            const BoundaryValues *bv, double dt, int32_t *isYielding, double *residual) {
  if (!ctx || !mk || !nf || !host || !mat || !opt || !bv) return FVM_ERR_ARG;
  FVM_TRY(fvm_grid_check(ctx, g));
  FVM_TRY(fvm_locate_async(ctx, g, mk, 0, mat, true));         // :243 + density :255-264
  int32_t y = 0;
  FVM_TRY(fvm_check_plastic_yielding(ctx, g, mk, mat, dt, &y, opt, 0.0));  // :299
  FVM_TRY(fvm_limit_viscosity(ctx, mk, opt));                   // :300
  FVM_TRY(fvm_project_markers_nodes_all2(ctx, g, mk, nf, mat)); // :303
  // host: formVEPSystem, KSP, retrieveSolutions, nodalStressStrain (:309-335)
  // Everything the calls below ask for is there: the passes run together.  An
  // empty store, two nodes along an axis or a missing array takes them one by one
  // (and a call that misses something says so at its place).
  const double *need[] = {host->dsxx,   host->dsyy,   host->dsxy,   host->soxx, host->soyy, host->soxy, host->edotxx,
                          host->edotxy, host->wxy,    host->p,      host->vx,   host->vy,   host->thisT, nf->lastT,
                          nf->rho,      nf->Cp,       nf->kThermal};
  bool all = mk->nMark > 0 && g->NX >= 3 && g->NY >= 3;
  for (const double *q : need) all = all && q != nullptr;
  if (all) {
    FVM_TRY(vep_after_stokes(ctx, g, mk, nf, host, mat, opt, bv, dt, residual));
    if (isYielding) *isYielding = y;
    return FVM_OK;
  }
  FVM_TRY(fvm_update_marker_strain_pressure(ctx, g, host, mk, mat, opt, dt));  // :341
  double r = 0.0;
  FVM_TRY(fvm_update_global_strain_rate_residual(ctx, g, mk, &r));            // :345
  if (opt->subgridStressDiffusivity > 0.0)                                      // :365
    FVM_TRY(fvm_subgrid_stress_changes(ctx, g, host, mk, mat, dt, opt->subgridStressDiffusivity));
  FVM_TRY(fvm_update_marker_stress(ctx, g, host, mk, mat));                     // :368
  NodalArrays th = *nf;  // subgrid T reads the projected lastT/rho/Cp/k
  FVM_TRY(fvm_subgrid_temperature_changes(ctx, host->thisT, g, &th, mk, mat, dt,  // :415
                                          opt->subgridTemperatureDiffusivity));
  NodalArrays adv = *host;
  FVM_TRY(fvm_advect_markers_rk(ctx, mk, &adv, g, bv, dt, ctx->jaumann));  // :435
  if (isYielding) *isYielding = y;
  if (residual) *residual = r;
  return FVM_OK;
}
