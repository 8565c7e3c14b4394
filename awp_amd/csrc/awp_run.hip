// Steps of the pmcl3d time loop on one Cartesian grid, NVE = 1
// (src/awp/pmcl3d.c:1628-2249): velocity, stress, point sources, stress
// imaging and receivers, launched from native code.
//
// Bound by the host on a small grid: a step of 64x64x64 keeps the GPU busy for
// 22 us, but assembling the arguments of its launches in Python took 47 us.
// The arguments change over a run only by the step's number, so a run passes
// them once: ten steps of 64x64x64 468 -> 225 us.
#include "awp_common.h"
#include "../../include/awp_hip.h"

extern "C" void awp_run_steps(const awp_run_t* R, int cur_step, int nsteps) {
  const char* W = "awp_run_steps";
  if (!R) {
    awp_set_error(AWP_ERR_ARG, "%s: null argument", W);
    return;
  }
  float* const* f = R->f;
  const hipStream_t St = (hipStream_t)R->stream;
  for (int n = cur_step + 1; n <= cur_step + nsteps; ++n) {
    dvelcx_H_opt(f[12], f[13], f[14], f[0], f[1], f[2], f[3], f[4], f[5], R->dcrjx, R->dcrjy,
                 R->dcrjz, R->d1, R->nyt, R->nzt, St, R->s_i, R->e_i, 0, 1);
#define AWP_RUN_STRESS(FN, ...)                                                                  \
  FN(f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], f[8], f[9], f[10], f[11], f[12], f[13],     \
     f[14], R->lam, R->mu, R->qp, R->coeff, R->qs, R->dcrjx, R->dcrjy, R->dcrjz, R->nyt, R->nzt, \
     St, R->lam_mu, __VA_ARGS__, R->nxt, R->NPC, 0, 0, R->s_i, R->e_i, R->s_j, R->e_j, 0)
    if (R->tex)
      AWP_RUN_STRESS(awp_dstrqc_tex, R->tex, R->ww);
    else if (R->newlit)
      AWP_RUN_STRESS(dstrqc_H_new, R->vx1, R->vx2, R->ww, R->wwo);
    else
      AWP_RUN_STRESS(dstrqc_H, R->vx1, R->vx2, R->ww, R->wwo);
#undef AWP_RUN_STRESS
    // sample n+1 of nst, as long as there is one (pmcl3d.c:2007-2015)
    if (R->nst && n < R->nst)
      addsrc_H(n + 1, R->nst, 3, R->psrc, R->npsrc, St, R->src[0], R->src[1], R->src[2],
               R->src[3], R->src[4], R->src[5], f[0], f[1], f[2], f[3], f[5], f[4], 0);
    fstr_H(f[2], f[4], f[5], St, R->s_i, R->e_i, R->s_j, R->e_j);
    if (n - 1 < R->rec_rows)
      awp_receivers_gather(f[12], f[13], f[14], R->rec_idx, R->rec_n, R->rec_out, n - 1, St, 0);
  }
}
