// sunhip_qseg.hip -- the pressure PCG's iteration on small and middle grids,
// one block per tile and one wave per segment of eight levels.
//
// Reference: CGSolveQ main/phys.c:2452-2524, OperatorQ :3486-3536,
// Preconditioner :3577-3619.
//
// With one lane walking a whole column (sunhip_q.hip) a grid of a few
// hundred tiles leaves most of the chip idle and every wave waits out one
// memory round trip per group of levels: 2000 columns of 50 levels took 44 us
// for the operator and 26 us for the preconditioner, whatever the bandwidth
// (12.7 and 8.7 us here, of which a launch alone is about 5).  Here a tile's
// columns are loaded by up to 8 waves at once:
//   apply    each wave forms qapply_tile's values on its segment's levels
//   precond  each wave updates r on its levels and holds them in registers
//            with l and the stored inverse pivots (qprec_tile's rows); the
//            two recurrences, a product and a difference per level, pass
//            from wave to wave
// and the block sums of each kernel are added by the blocks of the next one
// (as in the free-surface solve), so an iteration is two launches instead of
// four.  The values, the segment sums (SegSum) and the order in which tiles
// are added are those of the kernels in sunhip_q.hip: the same bits.
//
// The host launches at most QSEG_AHEAD iterations past the last one the
// device has reported (a word of pinned memory that each precond writes), so a
// solve ends with two or three idle iterations in the queue instead of up to
// two polling chunks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "sunhip_solvers.h"

using namespace sunhip;

namespace {

constexpr int QSEG_AHEAD = 2;

// The scalars a kernel runs on: in after its pending step on the sums of the
// kernel before (NV values per tile in part, in dispatch order), added as
// the group kernels and their finisher add them: four tiles of a group, 64
// groups by wave_sum, then the (at most 16) results in order.  load() issues
// the reads, so that they and the reads a caller issues after it are in
// flight together; finish() waits, adds, and has the first tile's block
// store the scalars to out with next_op pending unless the solve is done.
// Every block forms the same scalars.
template <int NV>
struct SegState {
  CGScal c;
  double p[2][NV][4];  // the first two chunks of 64 groups a wave adds
  __device__ __forceinline__ void load(const CGScal *in, const double *__restrict__ part, int nb4) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, W = blockDim.x >> 6;
    c = *in;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int v = (w + q * W) * 64 + l;
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < NV; i++) p[q][i][j] = v < nb4 ? part[(size_t)(v * 4 + j) * NV + i] : 0.0;
    }
  }
  // mu, nu and the iteration count; true when the solve is done
  __device__ __forceinline__ bool finish(CGScal *out, int nb4, const double *__restrict__ part, int next_op, bool first,
                                         double &mu, double &nu, int &iter, CGScal *host = nullptr) {
    __shared__ double sh[NV][16];
    __shared__ double sv[2];
    __shared__ int si[2];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, W = blockDim.x >> 6;
    for (int q = 0; w + q * W < 16; q++) {
      const int cq = w + q * W, v = cq * 64 + l;
#pragma unroll
      for (int i = 0; i < NV; i++) {
        double s = 0;
        if (cq * 64 < nb4) {
          if (v < nb4) {
            if (q == 0) {
#pragma unroll
              for (int j = 0; j < 4; j++) s += p[0][i][j];
            } else if (q == 1) {
#pragma unroll
              for (int j = 0; j < 4; j++) s += p[1][i][j];
            } else {
#pragma unroll
              for (int j = 0; j < 4; j++) s += part[(size_t)(v * 4 + j) * NV + i];
            }
          }
          s = wave_sum(s);
        }
        if (l == 0) sh[i][cq] = s;
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      if (c.pend && !c.done) {
        double tot[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) {
          double s = 0;
#pragma unroll
          for (int k = 0; k < 16; k++) s += sh[i][k];
          tot[i] = s;
        }
        q_op(&c, c.pend, tot);
      }
      sv[0] = c.mu; sv[1] = c.nu;
      si[0] = c.iter; si[1] = c.done;
      if (first) {
        c.pend = c.done ? 0 : next_op;
        *out = c;
        if (host) *host = c;
      }
    }
    __syncthreads();
    mu = sv[0]; nu = sv[1]; iter = si[0];
    return si[1] != 0;
  }
};

// The tile's share of NV dot products from its lanes' segment sums
// sh[i * 16 + segment][lane]: over the segments from the top, then over the
// lanes (valid in wave 0).
template <int NV>
__device__ void seg_block_sum(double (*sh)[64], int nseg, double (&tot)[NV]) {
  __syncthreads();
  if (threadIdx.x < 64)
#pragma unroll
    for (int i = 0; i < NV; i++) {
      double s = 0;
      for (int b = 0; b < nseg; b++) s += sh[i * 16 + b][threadIdx.x];
      tot[i] = wave_sum(s);
    }
}

// Segments g0 .. g1 - 1 of tile t in qapply_tile's FUSED or RESID mode, U
// levels at a time; the lane's sum of segment g goes to sh[g][lane].  A lane
// loads the groups its column reaches (at clamped addresses), and the first
// group's values are loaded before scalars() waits for the sums of the
// kernel before, which mu and nu come from.  Lanes past their column's bottom
// load nothing: clamped there, each would read its own last level, a cache
// line of its own per lane, face and field.  On columns of random depth an
// iteration of 512 tiles of 60 levels takes 58 us so, against 93 with every
// lane loading, 893 tiles 124 / 224; on smooth depths, 640 tiles of 70, 71 / 75.
// coef and dzf are read, not formed from the z-level windows: at these sizes
// they come from cache, and finding the windows costs as much as two
// iterations.
template <int MODE, int NF, int U, typename T, typename F>
__device__ __forceinline__ bool qapply_seg(const Geo &G, const QVec<T, T> &V, int t, int l, int g0, int g1,
                                           double (*sh)[64], F &&scalars) {
  constexpr bool FU = MODE == QM_FUSED;
  if (g0 >= g1) {  // below the tile's deepest column
    T a, b;
    return scalars(a, b);
  }
  const T *__restrict__ rt = FU ? V.rtmp : V.vin;
  const T *__restrict__ po = V.pold;
  const int s = t * 64 + l, NS = G.NS;
  const int n = G.nk[s], kt = G.ctop[s], nf = G.nf[s];
  const bool own = n > 0 && G.comp[s] == 1;
  const uint32_t base = n > 0 ? (uint32_t)(G.toff[t] + l) : 0u;
  uint32_t nbb[NF], ebb[NF];
  int kmn[NF], kmx[NF];
  T Df[NF];
#pragma unroll
  for (int f = 0; f < NF; f++) {
    // the per-face tables have SUNHIP_MAXF rows: load, then select
    const int nb = G.nbb[f * NS + s], eb = G.eb[f * NS + s], kr = G.kr[f * NS + s], es = G.es[f * NS + s];
    const T d = V.D[max(es, 0)];
    const bool on = own && f < nf && nb >= 0;
    nbb[f] = on ? (uint32_t)nb : base;
    ebb[f] = on ? (uint32_t)eb : 0u;
    kmn[f] = on ? (kr & 0xffff) : 0;
    kmx[f] = on ? (kr >> 16) : 0;
    Df[f] = on ? d : T(0);
  }
  T rv[U + 2], pv[U + 2], xv[U], nr[U][NF], np[U][NF], c[U + 1], dz[U][NF];
  // whether the lane has levels in the group at kb
  auto in = [&](int kb) { return own && kb < n && kb + U > kt; };
  auto load = [&](int kb) {
    if (!in(kb)) return;
#pragma unroll
    for (int j = 0; j < U + 2; j++) {  // levels kb - 1 .. kb + U
      const uint32_t idx = base + (uint32_t)min(max(kb - 1 + j, 0), n) * 64u;
      rv[j] = at32(rt, idx);
      pv[j] = FU ? at32(po, idx) : T(0);
      if (j > 0) c[j - 1] = at32(V.coef, idx);
    }
#pragma unroll
    for (int j = 0; j < U; j++) {
      const int k = kb + j;
      xv[j] = at32(FU ? (const T *)V.x : V.src, base + (uint32_t)min(k, n) * 64u);
#pragma unroll
      for (int f = 0; f < NF; f++) {
        const uint32_t kk = (uint32_t)min(k, max(kmx[f] - 1, 0)) * 64u;
        nr[j][f] = at32(rt, nbb[f] + kk);
        np[j][f] = FU ? at32(po, nbb[f] + kk) : T(0);
        dz[j][f] = at32(V.dzf, ebb[f] + kk);
      }
    }
  };
  load(g0 * SUNHIP_SEG);
  T mu = 0, nu = 0;
  if (FU && !scalars(mu, nu)) return false;
  double dot = 0;
  for (int kb = g0 * SUNHIP_SEG; kb < g1 * SUNHIP_SEG; kb += U) {
    if (kb > g0 * SUNHIP_SEG) load(kb);
    if (in(kb)) {
      T v[U + 2];
#pragma unroll
      for (int j = 0; j < U + 2; j++) v[j] = FU ? rv[j] + mu * pv[j] : rv[j];
#pragma unroll
      for (int j = 0; j < U; j++) {
        const int k = kb + j;
        if (k < kt || k >= n) continue;
        const T v0 = v[j + 1], vm1 = v[j], vp1 = v[j + 2], c0 = c[j], cp1 = c[j + 1];
        T y = 0;
#pragma unroll
        for (int f = 0; f < NF; f++) {
          const T nv = FU ? nr[j][f] + mu * np[j][f] : nr[j][f];
          const T term = (nv - v0) * dz[j][f] * Df[f];
          y = (k >= kmn[f] && k < kmx[f]) ? y + term : y;
        }
        if (kt == n - 1) y -= T(2.0) * c0 * v0;
        else if (k == kt) y += (-2 * c0 - cp1) * v0 + cp1 * vp1;
        else if (k == n - 1) y += c0 * vm1 - c0 * v0;
        else y += c0 * vm1 - (c0 + cp1) * v0 + cp1 * vp1;
        const uint32_t idx = base + (uint32_t)k * 64u;
        if (FU) {
          at32(V.pnew, idx) = v0;
          at32(V.x, idx) = xv[j] + nu * pv[j + 1];
          dot += (double)v0 * (double)y;
          at32(V.out, idx) = y;
        } else {
          at32(V.out, idx) = xv[j] - y;
        }
      }
    }
    if (FU && ((kb + U) & (SUNHIP_SEG - 1)) == 0) {
      sh[kb / SUNHIP_SEG][l] = dot;
      dot = 0;
    }
  }
  return true;
}

// The tile of block b (G.Nt and beyond: none) and its position in the group
// kernels' dispatch order, where its sums go.  Blocks are dealt to the 8
// XCDs round-robin; each XCD gets a contiguous run of groups of four tiles.
__device__ __forceinline__ int seg_tile(const Geo &G, int b, int &pos) {
  const int nb4 = (G.Nt + 3) >> 2, q = nb4 >> 3, r = nb4 & 7, x = b & 7, i = b >> 3;
  if ((i >> 2) >= q + (x < r ? 1 : 0)) return G.Nt;
  const int g = x * q + min(x, r) + (i >> 2), t = g * 4 + (i & 3);
  if (t < G.Nt) pos = G.b4perm[nb4 + g] * 4 + (t & 3);
  return t;
}

// Segments of the tile's deepest column.
__device__ __forceinline__ int seg_depth(const Geo &G, int t) {
  return (G.tdep[t] - 1 + SUNHIP_SEG - 1) / SUNHIP_SEG;
}

// The tile's sums at its position; the last tile also clears its group's
// positions past it.
template <int NV>
__device__ __forceinline__ void seg_put(const Geo &G, double *part, int t, int pos, const double (&tot)[NV]) {
#pragma unroll
  for (int i = 0; i < NV; i++) part[(size_t)pos * NV + i] = tot[i];
  if (t == G.Nt - 1)
    for (int j = (t & 3) + 1; j < 4; j++)
      for (int i = 0; i < NV; i++) part[(size_t)(pos - (t & 3) + j) * NV + i] = 0;
}

// spw segments per wave; MINW waves per SIMD
template <int NF, int U, int MINW, typename T>
__global__ __launch_bounds__(512, MINW) void k_qapply_seg(Geo G, QVec<T, T> V, const CGScal *sin, CGScal *sout,
                                                          const double *pin, double *pout, int nb4, int spw) {
  __shared__ double sh[16][64];
  int p = 0;
  const int t = seg_tile(G, blockIdx.x, p), w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (t >= G.Nt) return;
  const bool first = t == 0;
  SegState<2> St;
  St.load(sin, pin, nb4);
  auto scalars = [&](T &mu, T &nu) {
    double m, v;
    int iter;
    const bool done = St.finish(sout, nb4, pin, OP_APPLY, first, m, v, iter);
    mu = (T)m;
    nu = (T)v;
    return !done;
  };
  const int ns = seg_depth(G, t);
  if (!qapply_seg<QM_FUSED, NF, U, T>(G, V, t, l, w * spw, min(w * spw + spw, ns), sh, scalars)) return;
  double tot[1];
  seg_block_sum<1>(sh, ns, tot);
  if (threadIdx.x == 0) seg_put<1>(G, pout, t, p, tot);
}

// r = src - L x
template <int NF, int U, typename T>
__global__ __launch_bounds__(512) void k_qresid_seg(Geo G, QVec<T, T> V, int spw) {
  int p = 0;
  const int t = seg_tile(G, blockIdx.x, p), w = threadIdx.x >> 6;
  if (t >= G.Nt) return;
  qapply_seg<QM_RESID, NF, U, T>(G, V, t, threadIdx.x & 63, w * spw, min(w * spw + spw, seg_depth(G, t)), nullptr,
                                 [](T &, T &) { return true; });
}

// One or two (SPW) segments per wave, the waves in turn: every wave holds its
// levels' r, l and 1/b in registers, the forward recurrence passes from wave
// to wave through LDS (one value pair per column), then the backward one
// upward.  No level goes to memory or LDS between the sweeps.
// UPDATE: r -= nu z first.  Without it (the solve's first application) the
// scalars init are stored with OP_PREC_SETUP pending, and p0 and (x0 set) x
// are cleared.
template <bool UPDATE, int SPW, typename T>
__global__ __launch_bounds__(512, SPW == 1 ? 4 : 2) void k_qprec_seg(Geo G, const T *__restrict__ ql, const T *__restrict__ z,
                                                    T *__restrict__ r, T *__restrict__ out,
                                                    const T *__restrict__ bq, const CGScal *sin, CGScal *sout,
                                                    const double *pin, double *pout, int nb4, CGScal init, T *p0,
                                                    T *x0, unsigned long long *host, unsigned long long tag) {
  constexpr int SG = SUNHIP_SEG * SPW;
  __shared__ double sh[2 * 16][64];
  __shared__ T pass[2][64];
  int p = 0;
  const int t = seg_tile(G, blockIdx.x, p), w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (t >= G.Nt) return;
  const int nseg = seg_depth(G, t), W = (nseg + SPW - 1) / SPW;  // waves with levels
  SegState<1> St;
  if (UPDATE) {
    St.load(sin, pin, nb4);
    // to the host: the iterations completed before this one, and whether the
    // solve is done (first thing, so that the write is over before the kernel)
    if (t == 0 && threadIdx.x == 0)
      __hip_atomic_store(host, tag | ((unsigned long long)St.c.iter << 1) | (St.c.done ? 1u : 0u), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
  const int k0 = w * SG, s = t * 64 + l;
  const int n = G.nk[s], kt = G.ctop[s];
  const bool own = n > 0 && G.comp[s] == 1;
  const uint32_t base = n > 0 ? (uint32_t)(G.toff[t] + l) : 0u;
  T rn[SG], ib[SG], lv[SG], zv[SG];
  if (own && w < W && k0 < n && k0 + SG > kt) {  // the lane has levels here
#pragma unroll
    for (int j = 0; j < SG; j++) {
      const uint32_t idx = base + (uint32_t)min(k0 + j, n) * 64u;
      rn[j] = at32((const T *)r, idx);
      zv[j] = UPDATE ? at32(z, idx) : T(0);
      ib[j] = at32(bq, idx);
      lv[j] = at32(ql, idx);
    }
  }
  double mu = 0, nud = 0;
  int iter = 0;
  if (UPDATE) {
    if (St.finish(sout, nb4, pin, OP_PREC_ITER, t == 0, mu, nud, iter)) return;
  } else if (t == 0 && threadIdx.x == 0) {
    *sout = init;
  }
  const T nu = (T)nud;
  double rr[SPW] = {}, rz[SPW] = {};
#pragma unroll
  for (int j = 0; j < SG; j++) {
    const int k = k0 + j;
    const bool in = own && w < W && k >= kt && k < n;
    const T d = UPDATE ? rn[j] - nu * zv[j] : rn[j];
    rn[j] = in ? d : T(0);
    if (!in) { lv[j] = 0; ib[j] = 0; }
    if (UPDATE && in) at32(r, base + (uint32_t)k * 64u) = d;
    rr[j / SUNHIP_SEG] += (double)rn[j] * (double)rn[j];
  }
  // forward: d = r - l' d'; levels outside a column hold r = l = 0 and pass zeros on
  for (int b = 0; b < W; b++) {
    if (w == b) {
      T dp = b ? pass[0][l] : T(0), lp = b ? pass[1][l] : T(0);
#pragma unroll
      for (int j = 0; j < SG; j++) {
        dp = rn[j] - lp * dp;
        lp = lv[j];
        rn[j] = dp;
      }
      pass[0][l] = dp;
      pass[1][l] = lp;
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < SG; j++) {
    const T d = rn[j], e = d * ib[j];
    rz[j / SUNHIP_SEG] += (double)d * (double)e;
    rn[j] = e;
  }
  // backward: u = e - l u_below
  for (int b = W - 1; b >= 0; b--) {
    if (w == b) {
      T u = b < W - 1 ? pass[0][l] : T(0);
#pragma unroll
      for (int j = SG - 1; j >= 0; j--) {
        u = rn[j] - lv[j] * u;
        rn[j] = u;
      }
      pass[0][l] = u;
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < SG; j++) {
    const int k = k0 + j;
    if (own && k >= kt && k < n) {
      const uint32_t idx = base + (uint32_t)k * 64u;
      at32(out, idx) = rn[j];
      if (!UPDATE) {
        at32(p0, idx) = T(0);
        if (x0) at32(x0, idx) = T(0);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < SPW; q++)
    if (w * SPW + q < nseg) {
      sh[w * SPW + q][l] = rz[q];
      sh[16 + w * SPW + q][l] = rr[q];
    }
  double tot[2];
  seg_block_sum<2>(sh, nseg, tot);
  if (threadIdx.x == 0) seg_put<2>(G, pout, t, p, tot);
}

// The last iteration's step applied to the scalars (into sout and host),
// then (x set) x += nu p.
template <typename T>
__global__ __launch_bounds__(512) void k_qend_seg(Geo G, T *__restrict__ x, const T *__restrict__ p0,
                                                   const T *__restrict__ p1, const CGScal *sin, CGScal *sout,
                                                   const double *pin, int nb4, CGScal *host, int spw) {
  int p = 0;
  const int t = seg_tile(G, blockIdx.x, p), l = threadIdx.x & 63;
  if (t >= G.Nt) return;
  SegState<2> St;
  St.load(sin, pin, nb4);
  double mu, nu;
  int iter;
  St.finish(sout, nb4, pin, 0, t == 0, mu, nu, iter, host);
  if (!x || iter == 0) return;
  const T *__restrict__ pl = (iter & 1) ? p1 : p0;
  const int s = t * 64 + l, n = G.nk[s];
  if (n == 0 || G.comp[s] != 1) return;
  const uint32_t base = (uint32_t)(G.toff[t] + l);
  const int k0 = (threadIdx.x >> 6) * spw * SUNHIP_SEG, ka = max(k0, G.ctop[s]), kb = min(k0 + spw * SUNHIP_SEG, n);
  for (int k = ka; k < kb; k++) {
    const uint32_t idx = base + (uint32_t)k * 64u;
    at32(x, idx) = at32((const T *)x, idx) + (T)nu * at32(pl, idx);
  }
}

// Coefficients (DZZ: formed from the layer heights and stored, else read),
// inverse pivots and l of every column (qcoef_tile and qfactor_tile in one
// walk, eight levels' loads at a time).
template <typename T, bool DZZ>
__global__ __launch_bounds__(64) void k_qfactor_seg(Geo G, const double *__restrict__ dzz, T *__restrict__ coef,
                                                    T *__restrict__ bq, T *__restrict__ ql) {
  const int t = blockIdx.x, l = threadIdx.x, s = t * 64 + l, n = G.nk[s];
  if (n == 0) return;
  const int kt = G.ctop[s];
  const bool own = G.comp[s] == 1;
  const uint32_t base = (uint32_t)(G.toff[t] + l);
  const double Ac = DZZ ? G.Ac[s] : 0.0;
  constexpr int U = 8;
  double dprev = 0;
  T lprev = 0;
  for (int kb = kt; kb < n; kb += U) {
    T c[U + 1];
    if (DZZ) {
      double d[U + 1];
#pragma unroll
      for (int j = 0; j <= U; j++) d[j] = at32(dzz, base + (uint32_t)min(kb + j, n) * 64u);
#pragma unroll
      for (int j = 0; j <= U; j++) {
        c[j] = (T)(kb + j == kt ? Ac / d[j] : 2 * Ac / (d[j] + dprev));
        if (j < U && kb + j < n) at32(coef, base + (uint32_t)(kb + j) * 64u) = c[j];
        if (j < U) dprev = d[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j <= U; j++) c[j] = at32((const T *)coef, base + (uint32_t)min(kb + j, n) * 64u);
    }
    if (!own) continue;
#pragma unroll
    for (int j = 0; j < U; j++) {
      const int k = kb + j;
      if (k >= n) break;
      const T ck1 = k < n - 1 ? c[j + 1] : T(0);
      const T ib = kt == n - 1 ? T(-0.5) / c[j] : q_pivot<T>(k, kt, n, c[j], ck1, lprev);
      const T lk = ck1 * ib;
      at32(bq, base + (uint32_t)k * 64u) = ib;
      at32(ql, base + (uint32_t)k * 64u) = lk;
      lprev = lk;
    }
  }
}

int seg_count(const sunhip_grid *g) { return (g->maxdepth + SUNHIP_SEG - 1) / SUNHIP_SEG; }

// Segments per wave: the fewest with at most 8 waves per block and, where
// possible, every wave of the launch on the chip at once (16 per CU).
int seg_per_wave(const sunhip_grid *g, int most) {
  const int n = seg_count(g);
  int spw = (n + 7) / 8;
  while (spw < most && (int64_t)g->Nt * ((n + spw - 1) / spw) > 4096) spw++;
  return spw;
}

}  // namespace

namespace sunhip {

bool q_seg_ok(const sunhip_grid *g, const sunhip_cg_params *prm, size_t value_bytes) {
  // every knob of the one-lane-per-column kernels at its default
  const bool plain = g->tune_xchg < 0 && g->tune_tiles == 4 && !g->tune_blk && !g->tune_band && !g->tune_minw &&
                     g->tune_unroll == 4 && g->tune_nts && g->tune_rzid && g->tune_phead < 0 && g->tune_punroll == 8 &&
                     g->tune_reduce == 1;
  return plain && prm->precond == 2 && q_seg_fits(g, value_bytes);
}

bool q_seg_fits(const sunhip_grid *g, size_t value_bytes) {
  const bool size = g->Nt <= SUNHIP_QSEG_FULL ||
                    (g->Nt <= SUNHIP_QSEG_TILES && (size_t)g->Nflat * value_bytes <= SUNHIP_QSEG_BYTES);
  return g->tune_small && g->tune_order && size && seg_count(g) <= 16;
}

int q_seg_settle(sunhip_grid *g, CGScal *sc) {
  // one block reads all scalars before it writes them
  const int nb4 = (g->Nt + 3) / 4;
  k_qend_seg<double><<<1, 256, 0, g->stream>>>(g->geo(), nullptr, nullptr, nullptr, sc, sc, g->d_part + 4 * nb4, nb4,
                                               nullptr, 1);
  HIPCHK(hipGetLastError());
  return 0;
}

// Call fn<SPW> with the preconditioner's segments per wave.
template <typename F>
static void seg_launch(int spw, F &&fn) {
  if (spw == 1) fn(std::integral_constant<int, 1>{});
  else fn(std::integral_constant<int, 2>{});
}
// Register budget of the operator kernel, waves per SIMD: the most without spills.
constexpr int seg_minw(int nf) { return nf <= 3 ? 4 : nf == 4 ? 3 : 2; }
static int seg_blocks(const sunhip_grid *g) { return ((g->Nt + 3) / 4 + 7) / 8 * 32; }

int q_seg_setup64(sunhip_grid *g, const double *dzz, double *coef, double *bq, double *ql) {
  k_qfactor_seg<double, true><<<g->Nt, 64, 0, g->stream>>>(g->geo(), dzz, coef, bq, ql);
  HIPCHK(hipGetLastError());
  return 0;
}

int q_seg_factor32(sunhip_grid *g, float *coef, float *bq, float *ql) {
  k_qfactor_seg<float, false><<<g->Nt, 64, 0, g->stream>>>(g->geo(), nullptr, coef, bq, ql);
  HIPCHK(hipGetLastError());
  return 0;
}

int q_seg_resid64(sunhip_grid *g, const QVec<double, double> &V) {
  const int n = seg_count(g), spw = seg_per_wave(g, 4);
  with_nf(g->mf, [&](auto nfc) {
    constexpr int NF = decltype(nfc)::value;
    k_qresid_seg<NF, 2, double><<<seg_blocks(g), (n + spw - 1) / spw * 64, 0, g->stream>>>(g->geo(), V, spw);
    return 0;
  });
  HIPCHK(hipGetLastError());
  return 0;
}

template <typename T>
int q_seg_start(sunhip_grid *g, const sunhip_cg_params *prm, QSolver<T> &S, bool clear_x) {
  CGScal init{};
  init.tol = prm->epsilon;
  init.maxit = prm->maxiters;
  init.precond = prm->precond;
  init.resnorm = prm->resnorm;
  init.pend = OP_PREC_SETUP;
  const int nb4 = (g->Nt + 3) / 4, n = seg_count(g), pw = seg_per_wave(g, 2);
  double *prz = g->d_part + 4 * nb4;
  seg_launch(pw, [&](auto sp) {
    constexpr int SP = decltype(sp)::value;
    k_qprec_seg<false, SP, T><<<seg_blocks(g), (n + SP - 1) / SP * 64, 0, g->stream>>>(
        g->geo(), S.ql, nullptr, S.r, S.rtmp, S.bq, nullptr, S.sc, nullptr, prz, nb4, init, S.p0,
        clear_x ? S.x : nullptr, nullptr, 0);
  });
  HIPCHK(hipGetLastError());
  return 0;
}
template int q_seg_start<double>(sunhip_grid *, const sunhip_cg_params *, QSolver<double> &, bool);
template int q_seg_start<float>(sunhip_grid *, const sunhip_cg_params *, QSolver<float> &, bool);

template <typename T>
int q_seg_loop(sunhip_grid *g, const sunhip_cg_params *prm, QSolver<T> &S, int pk_apply, int pk_prec, bool finish) {
  const Geo G = g->geo();
  const int nb4 = (g->Nt + 3) / 4, nblk = seg_blocks(g), n = seg_count(g);
  const int spw = seg_per_wave(g, 4), pw = seg_per_wave(g, 2), W = (n + spw - 1) / spw;
  double *pz = g->d_part, *prz = g->d_part + 4 * nb4;
  volatile unsigned long long *word = g->h_prog;
  const unsigned long long tag = (unsigned long long)(++g->prog_tag & 0x7fffffff) << 32;
  auto seen = [&]() -> unsigned long long {
    const unsigned long long v = *word;
    return (v >> 32) == (tag >> 32) ? (v & 0xffffffffu) : 0;
  };
  for (int it = 0; it < prm->maxiters; it++) {
    unsigned long long v = seen();
    for (unsigned spin = 1; !(v & 1) && (int)(v >> 1) < it - QSEG_AHEAD; v = seen(), spin++) {
      if (spin % 4096) continue;
      const hipError_t e = hipStreamQuery(g->stream);  // nothing left that could report: go on
      if (e == hipSuccess) break;
      if (e != hipErrorNotReady) HIPCHK(e);
    }
    if (seen() & 1) break;
    QVec<T, T> V{};
    V.coef = S.coef; V.dzf = S.dzf; V.D = S.D; V.rtmp = S.rtmp; V.x = S.x; V.out = S.z;
    V.pold = (it & 1) ? S.p1 : S.p0;
    V.pnew = (it & 1) ? S.p0 : S.p1;
    int ps = prof_begin(g, pk_apply);
    with_nf(g->mf, [&](auto nfc) {
      constexpr int NF = decltype(nfc)::value;
      k_qapply_seg<NF, 2, seg_minw(NF), T><<<nblk, W * 64, 0, g->stream>>>(G, V, S.sc, S.sc + 1, prz, pz, nb4, spw);
      return 0;
    });
    prof_end(g, ps);
    ps = prof_begin(g, pk_prec);
    seg_launch(pw, [&](auto sp) {
      constexpr int SP = decltype(sp)::value;
      k_qprec_seg<true, SP, T><<<nblk, (n + SP - 1) / SP * 64, 0, g->stream>>>(G, S.ql, S.z, S.r, S.rtmp, S.bq, S.sc + 1,
                                                                              S.sc, pz, prz, nb4, CGScal{}, nullptr,
                                                                              nullptr, g->h_prog, tag);
    });
    prof_end(g, ps);
    HIPCHK(hipGetLastError());
  }
  // the settled scalars go to S.sc + 1 and the pinned copy the host reads
  k_qend_seg<T><<<finish ? nblk : 1, W * 64, 0, g->stream>>>(G, finish ? S.x : nullptr, S.p0, S.p1, S.sc, S.sc + 1, prz,
                                                             nb4, g->h_sc, spw);
  HIPCHK(hipGetLastError());
  return 0;
}
template int q_seg_loop<double>(sunhip_grid *, const sunhip_cg_params *, QSolver<double> &, int, int, bool);
template int q_seg_loop<float>(sunhip_grid *, const sunhip_cg_params *, QSolver<float> &, int, int, bool);

}  // namespace sunhip
