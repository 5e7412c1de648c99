// sunhip_solvers.h -- host-side pieces of the single-grid solvers that the
// batched engine (sunhip_batch.hip) reuses per member: set-up of one PCG
// (coefficients, pivots, initial residual, first preconditioned residual) and
// the final x update.  All of them only enqueue work on g->stream.
#pragma once
#include "sunhip_qtile.h"
#include "sunhip_htile.h"
#include "sunhip_tvdtile.h"
#include "sunhip_steptile.h"

namespace sunhip {

// Bytes of a cell field from which the iteration's seven vectors overflow the
// 256 MB memory-side cache, so that a launch's results are streamed.
#define SUNHIP_STREAM_BYTES (64 << 20)

// One pressure PCG instance: storage type, its scalars and its buffers.
template <typename T>
struct QSolver {
  CGScal *sc;
  const T *coef, *dzf, *D;
  T *x, *r, *z, *rtmp, *p0, *p1, *bq;
  const T *fcoef;  // qprecond=1: the scaled face coefficients
  ZReg Z;          // z-level windows of this solve (cwin null: none)
  T *ql;           // the rows' l (the iteration of sunhip_qseg.hip)
};

// One free-surface PCG instance.
template <typename T>
struct HSolver {
  CGScal *sc;
  const T *coef, *fcoef;
  T *x, *r, *z, *rt, *p0, *p1;
};

// The layer thicknesses dz[0..Nkmax) the z-level windows use (host array).
int set_zdz(sunhip_grid *g, const double *dz);
// The z-level windows of the pressure operator for the coefficients coef
// (FP64, from "dzz") and the face heights dzf now on the device; an empty
// ZReg when the layer thicknesses are unknown or the windows are switched
// off ("zreg" 0).
int q_windows(sunhip_grid *g, const double *coef, const double *dzf, ZReg *Z);

// The iteration of small and middle grids (sunhip_qseg.hip): one block per
// tile, with the defaults of the other kernels' knobs and qprecond=2.  It
// takes grids of at most SUNHIP_QSEG_FULL tiles, which the chip holds at once
// (two blocks per CU), and up to SUNHIP_QSEG_TILES while a field of the
// computational values is at most SUNHIP_QSEG_BYTES: a segment's stores and
// its reads of the levels above and below it miss the caches beyond that,
// where the whole-column kernels read each value once.  Per iteration,
// these kernels against those and their finishers, bathymetry of smooth bumps (0.55
// of the levels filled) or flat (all filled):
//   FP64  255 tiles of 40 levels 27 / 57 us, 508 of 70 52 / 84, 768 of 70 75 / 83,
//         254 of hexagons of 40 32 / 74; flat: 508 of 100 110 / 115, 508 of 128
//         143 / 158, 768 of 40 (15.8 MB) 64 / 66; but 768 of 70 (27 MB) 115 / 85,
//         996 of 40 (20.4 MB) 75 / 69, 996 of 100 (51 MB) 229 / 174
//         the line: 558 to 1000 tiles of 60 to 120 levels, any faces, 0.66 to
//         1.03 of the whole columns' time from 15.5 to 20 MB (of 48 levels
//         0.92 to 1.13), 0.72 to 1.33 to 24 MB, 0.9 to 1.5 beyond
//   FP32  508 of 70 40 / 83; flat: 996 of 40 (10 MB) 54 / 62, 996 of 70 (18 MB)
//         82 / 82, 996 of 100 (25 MB) 121 / 108
#define SUNHIP_QSEG_FULL 512
#define SUNHIP_QSEG_TILES 1024
#define SUNHIP_QSEG_BYTES 20000000
bool q_seg_ok(const sunhip_grid *g, const sunhip_cg_params *prm, size_t value_bytes);
// Whether the grid's size and dispatch order allow these kernels at all, for
// values of value_bytes each.
bool q_seg_fits(const sunhip_grid *g, size_t value_bytes);
// The scalars at sc after their pending first step (q_seg_start), in place.
int q_seg_settle(sunhip_grid *g, CGScal *sc);
// Coefficients, inverse pivots and l (QSolver::ql) from dzz, or the last two
// from FP32 coefficients.
int q_seg_setup64(sunhip_grid *g, const double *dzz, double *coef, double *bq, double *ql);
int q_seg_factor32(sunhip_grid *g, float *coef, float *bq, float *ql);
// V.out = V.src - L V.vin
int q_seg_resid64(sunhip_grid *g, const QVec<double, double> &V);
// rtmp = M^-1 r, p0 = 0 (and x = 0), fresh scalars with their first step pending.
template <typename T>
int q_seg_start(sunhip_grid *g, const sunhip_cg_params *prm, QSolver<T> &S, bool clear_x);
// Iterate until the device says done; the scalars then are in g->h_sc (after a
// wait for the stream) and at S.sc + 1, and (finish) x has its last update.
template <typename T>
int q_seg_loop(sunhip_grid *g, const sunhip_cg_params *prm, QSolver<T> &S, int pk_apply, int pk_prec, bool finish);

// Upload fresh CG scalars (tolerance, limits) to d from the pinned host slot
// stage (g->h_sc when null).  The slot must not be rewritten before the
// stream has executed the copy.
int upload_scal(sunhip_grid *g, CGScal *d, const sunhip_cg_params *prm, CGScal *stage = nullptr);

// Pressure solve, FP64, qprecond=2 or 0: everything up to the first iteration
// (main/phys.c:2441-2475) into the scalars at sc (g->d_qs when null).
int q_begin64(sunhip_grid *g, const sunhip_cg_params *prm, QSolver<double> *S, CGScal *stage, CGScal *sc = nullptr);
// x += nu*p of the last iteration.
int q_end64(sunhip_grid *g, const QSolver<double> &S);

// Mixed form: FP64 coefficients, FP32 copies of coef/dzf/D, FP32 pivots;
// S32 gets the FP32 PCG buffers (x = the correction e, scalars g->d_ms) and
// R the FP64 residual operands (out = the FP32 residual).  seg: for the
// iteration of sunhip_qseg.hip.
int q_mixed_prepare(sunhip_grid *g, const sunhip_cg_params *prm, QSolver<float> *S32, QVec<double, float> *R,
                    bool seg = false);
// Inner FP32 PCG from e = 0 on the residual already in S32.r.
int q_inner_begin(sunhip_grid *g, const sunhip_cg_params *inner, QSolver<float> &S32, CGScal *stage);
// The inner solve's last x update (scalars at sc), then x64 += e32.
int q_mix_finish(sunhip_grid *g, double *x, const QSolver<float> &S, const CGScal *sc);

// Free surface, FP64: coefficients, x = 0 on computational cells,
// r = b - L x, first preconditioned residual (main/phys.c:3108-3158).
int h_begin64(sunhip_grid *g, const sunhip_cg_params *prm, double grav, double theta, double dt,
              HSolver<double> *S, CGScal *stage);
int h_end64(sunhip_grid *g, const HSolver<double> &S);

// Arguments of one grid's scalar step (fields created on demand); no launch.
int tvd_args(sunhip_grid *g, const sunhip_scalar_params *sp, const char *scal, TvdArgs *T, ColArgs *C);

// Arguments of one grid's source / Corrector / Continuity stencils: qc, q and
// w name the correction, pressure and vertical velocity fields, src the
// source (fields created on demand); no launch.
int step_args(sunhip_grid *g, double theta, double dt, const char *qc, const char *q, const char *w,
              const char *src, StepArgs *out);

}  // namespace sunhip
