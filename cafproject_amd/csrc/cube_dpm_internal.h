/*
 * cube_dpm_internal.h -- state of one differentiable-PM box, shared by
 * cube_dpm.hip (the model) and cube_batch.hip (the ensemble runner).
 */
#ifndef CUBE_DPM_INTERNAL_H
#define CUBE_DPM_INTERNAL_H
#include "cube_internal.h"
#include "../../include/cube_dpm.h"

#define DPM_GMX 64 /* words that share the maximum of |g| */

struct cube_dpm {
  cube_dpm_params p;
  cube_ctx c; /* the stream, for the FFT layer */
  int64_t np, ng3, nf3, sg, sf; /* sg/sf: spectrum sizes (pitched) */
  int nb, nblk;         /* lattice blocks of 4^3 per axis and in all */
  int64_t npp;          /* particle slots, 64 per block */
  FFTPlan *plan_g, *plan_f;
  double ic[2];
  double *steps; /* host, 3*nsteps */
  float *amp;
  /* particle arrays: 3 floats per slot */
  float *xs, *ps;       /* positions (and momenta) of every `every`-th step */
  int every;
  float *xend, *xend_own; /* final positions: the last of xs, or an array of their own */
  float *x, *pw;        /* positions and momenta of recomputed steps */
  float *pm;            /* current momenta */
  float *xbar, *pbar;
  float *rho, *S, *lam;
  float *force;         /* the force mesh, or those of all steps (keep_force) */
  int keep_force;
  unsigned *gmx;        /* max |g| of the transpose's cotangents (float bits), two sets of DPM_GMX */
  int tile, ntile, tcap; /* cells per tile, tiles per axis, entries per list */
  int *tcnt, tpar;      /* two sets of list lengths, the one in use */
  uint32_t *tlist;
  uint64_t *trange;
  float2 *spec_f, *work3_f;
  float2 *spec_g, *work3_g;
  float *psi;           /* 3*ng^3 */
  int has_forward;
  int grid, block;      /* launch shape of the particle loops (tunable) */
};

#endif
