// sunhip_step.hip -- the stencils either side of the pressure solve on
// gfx950: the Poisson source (ComputeQSource, main/phys.c:2345-2395), the
// projection of the velocity and pressure (Corrector, main/phys.c:2301-2332)
// and the vertical velocity from continuity (Continuity,
// main/phys.c:3814-3844).  One launch each over max(Nt, Net) tiles: lanes
// of cell tiles own a column, lanes of edge tiles an edge.  The bodies live
// in sunhip_steptile.h, shared with the batched engine.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sunhip_steptile.h"
#include "sunhip_solvers.h"

using namespace sunhip;

// BAND: a wave per tile and band of levels (Bands), else one per tile.  The
// lock exchange (32 tiles of 50 levels): source 12.6 us, Corrector 53 -> 12.8,
// Continuity 70 -> 17.8.
template <int NF, bool BAND>
__global__ __launch_bounds__(256) void k_qsource(Geo G, StepArgs A, Bands B) {
  const int v = xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (!BAND) { qsource_tile<NF>(G, A, v, l); return; }
  const int t = v / B.nb, k0 = (v - t * B.nb) * B.len;
  qsource_tile<NF>(G, A, t, l, k0, k0 + B.len);
}

template <bool BAND>
__global__ __launch_bounds__(256) void k_corrector(Geo G, StepArgs A, Bands B) {
  const int v = xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (!BAND) { corrector_tile(G, A, v, l); return; }
  const int t = v / B.nb, k0 = (v - t * B.nb) * B.len;
  corrector_tile(G, A, t, l, k0, k0 + B.len);
}

// one block per tile, one wave per SUNHIP_SEG levels
template <int NF>
__global__ __launch_bounds__(1024) void k_continuity_seg(Geo G, StepArgs A) {
  __shared__ double carry[64];
  continuity_seg<NF>(G, A, xcd_block(blockIdx.x, gridDim.x), carry);
}

template <int NF>
__global__ __launch_bounds__(256) void k_continuity(Geo G, StepArgs A) {
  continuity_tile<NF>(G, A, xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
}

namespace sunhip {

// Device pointers of a step's fields (created on demand).  qc, q and w name
// the correction, the pressure and the vertical velocity fields; the others
// are fixed: u, utmp2, wtmp2, dzf, dzz, src, D.
int step_args(sunhip_grid *g, double theta, double dt, const char *qc, const char *q, const char *w,
              const char *src, StepArgs *out) {
  if (!g->have_extents) { set_error("time-step stencils: call sunhip_set_extents first"); return -1; }
  if (!(theta > 0) || !(dt > 0)) { set_error("time-step stencils: theta=%g and dt=%g must be positive", theta, dt); return -1; }
  Field *fu, *fw, *fq, *fqc, *fu2, *fw2, *fdzf, *fdzz, *fsrc, *fD;
  int rc = field(g, "u", &fu) | field(g, w, &fw) | field(g, q, &fq) | field(g, qc, &fqc) | field(g, "utmp2", &fu2) |
           field(g, "wtmp2", &fw2) | field(g, "dzf", &fdzf) | field(g, "dzz", &fdzz) | field(g, src, &fsrc) |
           field(g, "D", &fD);
  if (rc) return rc;
  if (fw->kind != CELLW || fw2->kind != CELLW) { set_error("time-step stencils: %s must be a w-type field", w); return -1; }
  if (fq->kind != CELL || fqc->kind != CELL || fsrc->kind != CELL) {
    set_error("time-step stencils: %s, %s and %s must be cell fields", q, qc, src);
    return -1;
  }
  StepArgs A{};
  A.u = fu->d; A.w = fw->d; A.q = fq->d; A.qc = fqc->d; A.utmp2 = fu2->d; A.wtmp2 = fw2->d; A.dzf = fdzf->d;
  A.dzz = fdzz->d; A.src = fsrc->d; A.D = fD->d; A.theta = theta; A.dt = dt;
  *out = A;
  return 0;
}

}  // namespace sunhip

extern "C" {

int sunhip_compute_qsource(sunhip_grid *g, double theta, double dt, const char *src) {
  HIPCHK(hipSetDevice(g->device));
  StepArgs A;
  int rc = step_args(g, theta, dt, "q", "qp", "w", src, &A);
  if (rc) return rc;
  const int tiles = std::max(g->Nt, g->Net), nb = (tiles + 3) / 4;
  const Bands B = level_bands(g, tiles);
  const int ps = prof_begin(g, PK_QSOURCE);
  with_nf(g->mf, [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    if (B.nb > 1) k_qsource<NF, true><<<(tiles * B.nb + 3) / 4, 256, 0, g->stream>>>(g->geo(), A, B);
    else k_qsource<NF, false><<<nb, 256, 0, g->stream>>>(g->geo(), A, B);
    return 0;
  });
  prof_end(g, ps);
  HIPCHK(hipGetLastError());
  return 0;
}

int sunhip_corrector(sunhip_grid *g, double dt, const char *qc, const char *q) {
  HIPCHK(hipSetDevice(g->device));
  StepArgs A;
  int rc = step_args(g, 1.0, dt, qc, q, "w", "src", &A);
  if (rc) return rc;
  const int tiles = std::max(g->Nt, g->Net);
  const Bands B = level_bands(g, tiles);
  const int ps = prof_begin(g, PK_CORRECT);
  if (B.nb > 1) k_corrector<true><<<(tiles * B.nb + 3) / 4, 256, 0, g->stream>>>(g->geo(), A, B);
  else k_corrector<false><<<(tiles + 3) / 4, 256, 0, g->stream>>>(g->geo(), A, B);
  prof_end(g, ps);
  HIPCHK(hipGetLastError());
  return 0;
}

int sunhip_continuity(sunhip_grid *g, double theta, const char *w) {
  HIPCHK(hipSetDevice(g->device));
  StepArgs A;
  int rc = step_args(g, theta, 1.0, "q", "qp", w, "src", &A);
  if (rc) return rc;
  const Geo G = g->geo();
  const int nb = (g->Nt + 3) / 4;
  const int ps = prof_begin(g, PK_CONTINUITY);
  const int ns = (g->maxdepth + SUNHIP_SEG - 1) / SUNHIP_SEG;
  with_nf(g->mf, [&](auto nf) {
    constexpr int NF = decltype(nf)::value;
    if constexpr (NF <= 4)
      if (g->tune_small && g->Nt <= 1024 && ns <= 16) {
        k_continuity_seg<NF><<<g->Nt, ns * 64, 0, g->stream>>>(G, A);
        return 0;
      }
    k_continuity<NF><<<nb, 256, 0, g->stream>>>(G, A);
    return 0;
  });
  prof_end(g, ps);
  HIPCHK(hipGetLastError());
  return 0;
}

}  // extern "C"
