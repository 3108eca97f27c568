// Multigrid-preconditioned conjugate gradients for the systems of meshes:
// FP64 CG on the Dirichlet-eliminated matrix, its preconditioner one V-cycle
// over a hierarchy of uniform grids.
//
// Jacobi-PCG takes O(1/h) iterations (4,800 at 1024^2); the V-cycle keeps the
// count at 13 - 16 for P1 at every size (P2: 16 - 27), so a solve reads the
// matrix about 60 times in all.  One forward + adjoint on MI355X, Jacobi-PCG
// -> this: Poisson 64^2 FP64 9.1 -> 1.7 ms, 511^2 FP64 81 -> 3.6 ms, 1024^2
// mixed 276 -> 5.9 ms, heat 200^2 16.5 -> 2.4 ms, P2 101^2 43 -> 4.7 ms; the
// small ones are bound by launches (about 5 us each), the large ones by the
// fine level's passes over memory.  The grids are laid over the mesh's bounding box (cells of about
// four rows) and know nothing of the triangles: a row takes part through the
// bilinear interpolation P from the four nodes of its cell, and every coarse
// matrix is the Galerkin product P^T A P of the assembled matrix, a 25-point
// stencil on each grid, so boundary conditions, holes, coefficients and mass
// terms need no special case.  Rows of Dirichlet nodes are not interpolated.
//
// Smoother: x += w M^-1 (b - A x) with M_ii = a_ii sum_j |a_ij| /
// sqrt(a_ii a_jj) (the l1 row sums of the diagonally scaled matrix): M - A/1
// is positive semidefinite for every SPD A, so with w < 2 the V-cycle is SPD
// and CG's convergence theory holds whatever the mesh (Baker, Falgout, Kolev
// & Yang 2011 for the l1 smoothers; the scaled sums keep grid nodes that
// barely touch the mesh from dominating their neighbours').
//
// Precision: the matrix, residual, direction, solution and every dot product
// of CG are FP64.  The V-cycle works on FP32 copies (fine level: the scaled
// form S A S of cg.hip) with FP64 sums; it only shapes the search direction.
// A solve is converged when the residual recomputed from the FP64 matrix is.
//
// One iteration (every kernel returns at once when its system is done):
//   mk_dir     p = z + beta p, q = A p; partials of p.q, r.q, q.q, r.r
//   ms_alpha   alpha = r.z / p.q and the new |r|^2 = r.r - 2 alpha r.q +
//              alpha^2 q.q
//   mk_update  x += alpha p, r -= alpha q, first smoothing step from zero
//   mk_res     residual of that, mk_restrict to the first grid (with its
//              first smoothing step)
//   gk_*       the grids down to MG_TAIL nodes: residual, restriction
//   mk_tail    the remaining grids, one workgroup per system, in LDS
//   gk_*       and up: prolongation, smoothing
//   mk_prolong, mk_post  the fine level's; z, partials of r.z
//   ms_beta    beta = r.z / previous r.z
// No atomics, no fences; every reduction has one order.
#include <hipcub/hipcub.hpp>

#include <chrono>
#include <cmath>

#include "batched.h"
#include "geom.h"
#include "mg.h"
#include "sell.h"

namespace admfem {

namespace {

constexpr int NT = 256;   // threads of the wide kernels
constexpr int RT = 1024;  // threads of the one-block kernels
constexpr int ST_RUN = 0, ST_CONV = 1, ST_MAXIT = 2, ST_NAN = 3, ST_BREAK = 4;
// Smoothing weight: any value below 2 is safe; 1.6 took the fewest
// iterations over jittered meshes (15 with 4/3, 13 - 14 with 1.5 - 1.7).
constexpr float OM = 1.6f;

inline unsigned nb(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// The system and block of a grid block: from the batch's map, or (no map)
// system `sys` with the blocks dealt to the 8 XCDs in contiguous eighths.
__device__ __forceinline__ int2 where(const int2 *map, int sys) {
  if (map) return map[blockIdx.x];
  return make_int2(sys, xcd_block(blockIdx.x, gridDim.x));
}

typedef float f2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ gptr<f2_t> frac_ptr(const MgSys &d) {
  return (gptr<f2_t>)reinterpret_cast<const f2_t *>(d.frac);
}

template <int NV>
__device__ __forceinline__ void put_partials(const double (&v)[NV], double *part, int G,
                                             int lb) {
  __shared__ double sh[NV][NT / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const double t = wave_sum(v[j]);
    if (lane == 0) sh[j][wv] = t;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < NT / 64; k++) t += sh[threadIdx.x][k];
    global_mut(part)[(size_t)threadIdx.x * G + lb] = t;
  }
}

// One block's sums of NV partial arrays of length G (fixed order).
template <int NV>
__device__ __forceinline__ void sum_partials(const double *part_, int G, double (&out)[NV]) {
  __shared__ double sh[NV][RT / 64];
  const gptr<double> part = global_ptr(part_);
  double a[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) a[j] = 0.0;
  int k = threadIdx.x;
  for (; k + 3 * RT < G; k += 4 * RT) {
    double v[NV][4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < NV; j++) v[j][u] = part[(size_t)j * G + k + u * RT];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < NV; j++) a[j] += v[j][u];
  }
  for (; k < G; k += RT)
#pragma unroll
    for (int j = 0; j < NV; j++) a[j] += part[(size_t)j * G + k];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const double t = wave_sum(a[j]);
    if (lane == 0) sh[j][wv] = t;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NV; j++) {
    double t = 0.0;
#pragma unroll
    for (int k2 = 0; k2 < RT / 64; k2++) t += sh[j][k2];
    out[j] = t;
  }
}

// ------------------------------------------------------ per-matrix set-up

// dsq = 1/sqrt(a_ii), sq = sqrt(a_ii), the FP32 scaled off-diagonals and the
// smoother's weights.  A row without a positive diagonal (an isolated node,
// or a matrix that is not SPD) gets weight 0: the preconditioner skips it.
__global__ void __launch_bounds__(NT)
    mk_scale(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  const gptr<double> dg = global_ptr(d.diag), sv = global_ptr(d.sv64);
  const gptr<int> sc = global_ptr(d.sc), sp = global_ptr(d.sp);
  const double aii = dg[i];
  const double si = aii > 0.0 ? 1.0 / sqrt(aii) : 0.0;
  global_mut(d.dsq)[i] = si;
  global_mut(d.sq)[i] = aii > 0.0 ? (float)sqrt(aii) : 0.0f;
  const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
  double sum = 1.0;
  for (int k = 0; k < w; k++) {
    const int e = off + 64 * k;
    const double ajj = dg[sc[e]];
    const float v = ajj > 0.0 ? (float)(sv[e] * si * (1.0 / sqrt(ajj))) : 0.0f;
    global_mut(d.sv32)[e] = v;
    sum += fabs((double)v);
  }
  global_mut(d.minv)[i] = aii > 0.0 ? (float)(1.0 / sum) : 0.0f;
}

// The first grid's matrix P^T A P: one thread per grid node, gathering from
// the rows of its four cells; the 25 sums of a thread live in LDS (they are
// addressed by the columns' cells).
constexpr int GT = 128;
__global__ void __launch_bounds__(GT)
    mk_galerkin(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys) {
  __shared__ double acc[25][GT];
  const int2 mb = where(map, sys);
  if (mb.x < 0) return;
  const MgSys &d = D[mb.x];
  const MgLevel &l = d.lv[0];
  const int id = mb.y * GT + threadIdx.x, tid = threadIdx.x;
  if (id >= l.nx * l.ny) return;
  const int X = id % l.nx, Y = id / l.nx, ncx = l.nx - 1, ncy = l.ny - 1;
#pragma unroll
  for (int o = 0; o < 25; o++) acc[o][tid] = 0.0;
  const gptr<int> cptr = global_ptr(d.cptr), crow = global_ptr(d.crow), cell = global_ptr(d.cell);
  const gptr<int> sc = global_ptr(d.sc), sp = global_ptr(d.sp);
  const gptr<double> sv = global_ptr(d.sv64), dg = global_ptr(d.diag);
  const gptr<f2_t> frac = frac_ptr(d);
  for (int cy = max(Y - 1, 0); cy <= min(Y, ncy - 1); cy++) {
    const int c0 = cy * ncx + max(X - 1, 0), c1 = cy * ncx + min(X, ncx - 1);
    for (int k = cptr[c0]; k < cptr[c1 + 1]; k++) {
      const int i = crow[k], ci = cell[i];
      const f2_t f = frac[i];
      const double wi = (double)(ci - cy * ncx == X ? 1.0f - f.x : f.x) *
                        (double)(cy == Y ? 1.0f - f.y : f.y);
      const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
      for (int e = -1; e < w; e++) {
        const int j = e < 0 ? i : sc[off + 64 * e];
        const double v = wi * (e < 0 ? dg[i] : sv[off + 64 * e]);
        const int cj = cell[j];
        if (cj < 0) continue;
        const f2_t g = frac[j];
        const int ox = cj % ncx - X + 2, oy = cj / ncx - Y + 2;
        if (ox < 0 || ox > 3 || oy < 0 || oy > 3) continue;  // (the plan excludes these)
        acc[oy * 5 + ox][tid] += v * ((1.0 - g.x) * (1.0 - g.y));
        acc[oy * 5 + ox + 1][tid] += v * ((double)g.x * (1.0 - g.y));
        acc[oy * 5 + ox + 5][tid] += v * ((1.0 - g.x) * (double)g.y);
        acc[oy * 5 + ox + 6][tid] += v * ((double)g.x * (double)g.y);
      }
    }
  }
  const int at = mg_at(l.px, X, Y);
#pragma unroll
  for (int o = 0; o < 25; o++) global_mut(l.a)[(size_t)o * l.pn + at] = (float)acc[o][tid];
}

// One node's entries of the next grid's matrix: P^T A P with the bilinear
// interpolation of a grid from every second node.
__device__ __forceinline__ void coarse_node(const MgLevel &f, const MgLevel &c, int X, int Y) {
  double T[7][7];
#pragma unroll
  for (int u = 0; u < 7; u++)
#pragma unroll
    for (int v = 0; v < 7; v++) T[u][v] = 0.0;
  const gptr<float> a = global_ptr(f.a);
#pragma unroll
  for (int dy = -1; dy <= 1; dy++)
#pragma unroll
    for (int dx = -1; dx <= 1; dx++) {
      const int x = 2 * X + dx, y = 2 * Y + dy;
      if (x < 0 || y < 0 || x >= f.nx || y >= f.ny) continue;
      const double w = (dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0);
      const int at = mg_at(f.px, x, y);
#pragma unroll
      for (int oy = 0; oy < 5; oy++)
#pragma unroll
        for (int ox = 0; ox < 5; ox++)
          T[dy + oy + 1][dx + ox + 1] += w * (double)a[(size_t)(oy * 5 + ox) * f.pn + at];
    }
  const int at = mg_at(c.px, X, Y);
#pragma unroll
  for (int oy = -2; oy <= 2; oy++)
#pragma unroll
    for (int ox = -2; ox <= 2; ox++) {
      double s = 0.0;
#pragma unroll
      for (int v = -1; v <= 1; v++)
#pragma unroll
        for (int u = -1; u <= 1; u++) {
          const int ty = 2 * oy + v + 3, tx = 2 * ox + u + 3;
          if (ty >= 0 && ty < 7 && tx >= 0 && tx < 7)
            s += (u ? 0.5 : 1.0) * (v ? 0.5 : 1.0) * T[ty][tx];
        }
      global_mut(c.a)[(size_t)((oy + 2) * 5 + ox + 2) * c.pn + at] = (float)s;
    }
}

// A grid's smoothing weights.
__device__ __forceinline__ void weight_node(const MgLevel &l, int x, int y) {
  const gptr<float> a = global_ptr(l.a);
  const int at = mg_at(l.px, x, y);
  const float aii = a[(size_t)12 * l.pn + at];
  double s = 0.0;
#pragma unroll
  for (int o = 0; o < 25; o++) {
    const float v = a[(size_t)o * l.pn + at];
    const float ajj = a[(size_t)12 * l.pn + at + (o / 5 - 2) * l.px + o % 5 - 2];
    if (ajj > 0.0f) s += fabs((double)v) / sqrt((double)ajj);
  }
  global_mut(l.minv)[at] = aii > 1e-30f ? (float)(1.0 / (sqrt((double)aii) * s)) : 0.0f;
}

__global__ void __launch_bounds__(GT)
    gk_galerkin(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys, int k) {
  const int2 mb = where(map, sys);
  if (mb.x < 0) return;
  const MgLevel &f = D[mb.x].lv[k - 1], &c = D[mb.x].lv[k];
  const int id = mb.y * GT + threadIdx.x;
  if (id < c.nx * c.ny) coarse_node(f, c, id % c.nx, id / c.nx);
}

__global__ void __launch_bounds__(GT)
    gk_weights(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys, int k) {
  const int2 mb = where(map, sys);
  if (mb.x < 0) return;
  const MgLevel &l = D[mb.x].lv[k];
  const int id = mb.y * GT + threadIdx.x;
  if (id < l.nx * l.ny) weight_node(l, id % l.nx, id / l.nx);
}

// The tail's grids (from d.tail on, whose matrix is there) and the dense
// inverse of the last one by Gauss-Jordan on its scaled form; a node whose
// pivot vanishes (outside the mesh, or the constant of a singular matrix)
// is left out.
constexpr int ST = 512;  // (each thread holds a 7 x 7 patch)
__global__ void __launch_bounds__(ST)
    mk_tail_setup(const MgSys *__restrict__ D, const int *__restrict__ list, int sys) {
  if (list) sys = list[blockIdx.x];
  if (sys < 0) return;
  const MgSys &d = D[sys];
  for (int k = d.tail; k < d.nlev; k++) {
    const MgLevel &l = d.lv[k];
    const int nn = l.nx * l.ny;
    if (k > d.tail) {
      for (int id = threadIdx.x; id < nn; id += ST) coarse_node(d.lv[k - 1], l, id % l.nx, id / l.nx);
      __syncthreads();
    }
    for (int id = threadIdx.x; id < nn; id += ST) weight_node(l, id % l.nx, id / l.nx);
    __syncthreads();
  }
  __shared__ double A[MG_DENSE][MG_DENSE + 1], sc[MG_DENSE], col[MG_DENSE];
  const MgLevel &l = d.lv[d.nlev - 1];
  const int nn = l.nx * l.ny;
  const gptr<float> a = global_ptr(l.a);
  for (int i = threadIdx.x; i < nn; i += ST) {
    const float aii = a[(size_t)12 * l.pn + mg_at(l.px, i % l.nx, i / l.nx)];
    sc[i] = aii > 1e-30f ? 1.0 / sqrt((double)aii) : 0.0;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < nn * nn; t += ST) {
    const int i = t / nn, j = t % nn;
    const int dx = j % l.nx - i % l.nx, dy = j / l.nx - i / l.nx;
    double v = 0.0;
    if (abs(dx) <= 2 && abs(dy) <= 2)
      v = (double)a[(size_t)((dy + 2) * 5 + dx + 2) * l.pn + mg_at(l.px, i % l.nx, i / l.nx)];
    A[i][j] = v * sc[i] * sc[j];
  }
  __syncthreads();
  for (int k = 0; k < nn; k++) {
    const double pv = A[k][k];
    const bool skip = !(pv > 1e-9);
    for (int i = threadIdx.x; i < nn; i += ST) col[i] = A[i][k];
    __syncthreads();
    if (skip) {  // the variable leaves the system: zero row and column
      for (int t = threadIdx.x; t < nn; t += ST) {
        A[t][k] = 0.0;
        A[k][t] = 0.0;
      }
    } else {
      for (int t = threadIdx.x; t < nn; t += ST)
        if (t != k) A[k][t] /= pv;
      __syncthreads();
      for (int t = threadIdx.x; t < nn * nn; t += ST) {
        const int i = t / nn, j = t % nn;
        if (i != k && j != k) A[i][j] -= col[i] * A[k][j];
      }
      __syncthreads();
      for (int t = threadIdx.x; t < nn; t += ST) A[t][k] = t == k ? 1.0 / pv : -col[t] / pv;
    }
    __syncthreads();
  }
  for (int t = threadIdx.x; t < nn * nn; t += ST) {
    const int i = t / nn, j = t % nn;
    global_mut(d.cinv)[t] = (float)(A[i][j] * sc[i] * sc[j]);
  }
}

// The smallest row sum over diagonal of the interior rows (per block, then
// over the blocks): what the mass term leaves of the constant's energy.
__global__ void __launch_bounds__(NT)
    mk_rowsum(int n, const int *__restrict__ row_bd, const int *__restrict__ sp,
              const double *__restrict__ sv, const double *__restrict__ diag,
              double *__restrict__ out) {
  const int i = blockIdx.x * NT + threadIdx.x;
  double v = 1.0;
  if (i < n && row_bd[i] < 0) {
    const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
    double sum = diag[i];
    for (int k = 0; k < w; k++) sum += sv[off + 64 * k];
    v = sum / diag[i];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  __shared__ double sh[NT / 64];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < NT / 64; k++) v = fmin(v, sh[k]);
    out[1 + blockIdx.x] = v;
  }
}
__global__ void __launch_bounds__(RT) ms_rowsum(int G, double *__restrict__ out) {
  double v = 1.0;
  for (int k = threadIdx.x; k < G; k += RT) v = fmin(v, out[1 + k]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  __shared__ double sh[RT / 64];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < RT / 64; k++) v = fmin(v, sh[k]);
    out[0] = v;
  }
}

__global__ void mk_zero(float *__restrict__ a, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.0f;
}

// ---------------------------------------------------------------- CG kernels

// The scaled residual and the first smoothing step (from zero) of a row.
__device__ __forceinline__ void first_smooth(const MgSys &d, int i, double ri) {
  const float rs = (float)(ri * global_ptr(d.dsq)[i]);
  global_mut(d.rs)[i] = rs;
  global_mut(d.x0)[i] = OM * global_ptr(d.minv)[i] * rs;
}

// Row i's product with the FP32 scaled off-diagonals.
template <class L>
__device__ __forceinline__ double dot32(const MgSys &d, int i, L load) {
  auto dbl = [](float v) { return (double)v; };
  return d.sd ? sell_dot16<float>(i, d.sp, d.sd, d.sv32, load, dbl)
              : sell_dot<float>(i, d.sp, d.sc, d.sv32, load, dbl);
}

// Start: x = b on identity rows and 0 elsewhere, r = b - A x (0 on those
// rows, b on the rest), p = 0.  Restart (FRESH false): r = b - A x of the
// current x.  Partials of r.r and b.b.  (b_ null: the descriptor's b.)
template <bool FRESH>
__global__ void __launch_bounds__(NT)
    mk_start(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys,
             const double *b_) {
  const int2 m = where(map, sys);
  if (m.x < 0) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  double t[2] = {0.0, 0.0};
  if (i < d.npad) {
    const double bi = i < d.n ? global_ptr(b_ ? b_ : d.b)[i] : 0.0;
    double ri;
    if (FRESH) {
      const bool ident = i >= d.n || global_ptr(d.row_bd)[i] >= 0;
      ri = ident ? 0.0 : bi;
      global_mut(d.x)[i] = (ident && i < d.n) ? bi : 0.0;
      global_mut(d.p[0])[i] = 0.0;
      global_mut(d.p[1])[i] = 0.0;
    } else {
      const gptr<double> x = global_ptr(d.x);
      const double ax = global_ptr(d.diag)[i] * x[i] +
                        sell_dot<double>(i, d.sp, d.sc, d.sv64, [&](int c) { return x[c]; });
      ri = bi - ax;
    }
    global_mut(d.r)[i] = ri;
    first_smooth(d, i, ri);
    t[0] = ri * ri;
    t[1] = bi * bi;
  }
  put_partials<2>(t, d.part, d.nblk, m.y);
}

__global__ void __launch_bounds__(RT)
    ms_start(const MgSys *__restrict__ D, MgScal *S_, int sys, int fresh, double rtol2,
             int maxit) {
  const MgSys &d = D[sys];
  MgScal *S = S_ + sys;
  double t[2];
  sum_partials<2>(d.part, d.nblk, t);
  if (threadIdx.x != 0) return;
  if (fresh) {
    S->rtol2 = rtol2;
    S->bb = t[1];
    S->tol2 = rtol2 * t[1];
    S->it = 0;
    S->maxit = maxit;
    S->nrepl = 0;
  } else {
    S->nrepl += 1;
  }
  S->rr = t[0];
  S->rz = 0.0;
  S->alpha = S->beta = 0.0;
  S->first = 1;
  S->apply = 0;
  S->status = (!(t[0] == t[0]) || !isfinite(t[0])) ? ST_NAN
              : t[0] <= S->tol2                    ? ST_CONV
              : S->it >= S->maxit                  ? ST_MAXIT
                                                   : ST_RUN;
}

// p = z + beta p (into the other buffer), q = A p; partials of p.q, r.q,
// q.q, r.r.  A neighbour's p is formed on the fly by the same fused
// multiply-add as its own row forms it.
__global__ void __launch_bounds__(NT)
    mk_dir(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const double beta = S[m.x].beta;
  const bool odd = S[m.x].it & 1;
  const gptr<double> p = global_ptr(d.p[odd]);
  const gptr<float> z = global_ptr(d.z);
  const int i = m.y * NT + threadIdx.x;
  double t[4] = {0.0, 0.0, 0.0, 0.0};
  if (i < d.npad) {
    struct zp { float z; double p; };
    auto load = [&](int c) { return zp{z[c], p[c]}; };
    auto comb = [&](zp v) { return fma(beta, v.p, (double)v.z); };
    const double pi = comb(load(i)), ri = global_ptr(d.r)[i];
    const double qi = global_ptr(d.diag)[i] * pi + sell_dot<double>(i, d.sp, d.sc, d.sv64, load, comb);
    global_mut(d.p[!odd])[i] = pi;
    global_mut(d.q)[i] = qi;
    t[0] = pi * qi;
    t[1] = ri * qi;
    t[2] = qi * qi;
    t[3] = ri * ri;
  }
  put_partials<4>(t, d.part, d.nblk, m.y);
}

__global__ void __launch_bounds__(RT)
    ms_alpha(const MgSys *__restrict__ D, MgScal *S_, const int *__restrict__ list, int sys) {
  if (list) sys = list[blockIdx.x];
  MgScal *S = S_ + sys;
  if (S->status != ST_RUN) {
    if (threadIdx.x == 0) S->apply = 0;
    return;
  }
  double t[4];
  sum_partials<4>(D[sys].part, D[sys].nblk, t);
  if (threadIdx.x != 0) return;
  const double pq = t[0];
  S->apply = 0;
  S->it += 1;
  if (pq != pq || !isfinite(pq)) {
    S->status = ST_NAN;
  } else if (!(pq > 0.0)) {
    S->status = ST_BREAK;  // not SPD
  } else {
    const double alpha = S->rz / pq;
    S->alpha = alpha;
    S->rr = fmax(t[3] - 2.0 * alpha * t[1] + alpha * alpha * t[2], 0.0);
    S->apply = 1;
    if (S->rr <= S->tol2) S->status = ST_CONV;
    else if (S->it >= S->maxit) S->status = ST_MAXIT;
  }
}

// x += alpha p, r -= alpha q, first smoothing step (p: the buffer mk_dir
// wrote, after ms_alpha has counted the step)
__global__ void __launch_bounds__(NT)
    mk_update(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
              int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || !S[m.x].apply) return;
  const MgSys &d = D[m.x];
  const double alpha = S[m.x].alpha;
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  const double pi = global_ptr(d.p[S[m.x].it & 1])[i];
  const double xi = fma(alpha, pi, global_ptr(d.x)[i]);
  const double ri = fma(-alpha, global_ptr(d.q)[i], global_ptr(d.r)[i]);
  global_mut(d.x)[i] = xi;
  global_mut(d.r)[i] = ri;
  first_smooth(d, i, ri);
}

// t = the fine residual after the first smoothing step, in the unscaled
// form's dual times the interpolation's weight: sqrt(a_ii) (rs - Â x0)
__global__ void __launch_bounds__(NT)
    mk_res(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  const gptr<float> x0 = global_ptr(d.x0);
  const double res = (double)global_ptr(d.rs)[i] - (double)x0[i] -
                     dot32(d, i, [&](int c) { return x0[c]; });
  global_mut(d.t)[i] = (float)(res * (double)global_ptr(d.sq)[i]);
}

// First grid: b = P^T t and the first smoothing step from zero.
__global__ void __launch_bounds__(NT)
    mk_restrict(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
                int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const MgLevel &l = d.lv[0];
  const int id = m.y * NT + threadIdx.x;
  if (id >= l.nx * l.ny) return;
  const int X = id % l.nx, Y = id / l.nx, ncx = l.nx - 1, ncy = l.ny - 1;
  const gptr<int> cptr = global_ptr(d.cptr), crow = global_ptr(d.crow), cell = global_ptr(d.cell);
  const gptr<float> t = global_ptr(d.t);
  const gptr<f2_t> frac = frac_ptr(d);
  double s = 0.0;
  for (int cy = max(Y - 1, 0); cy <= min(Y, ncy - 1); cy++) {
    const int c0 = cy * ncx + max(X - 1, 0), c1 = cy * ncx + min(X, ncx - 1);
    const int k1 = cptr[c1 + 1];
    for (int k = cptr[c0]; k < k1; k++) {
      const int i = crow[k];
      const f2_t f = frac[i];
      s += (double)((cell[i] - cy * ncx == X ? 1.0f - f.x : f.x) *
                    (cy == Y ? 1.0f - f.y : f.y)) * (double)t[i];
    }
  }
  const int at = mg_at(l.px, X, Y);
  global_mut(l.b)[at] = (float)s;
  global_mut(l.x)[at] = OM * global_ptr(l.minv)[at] * (float)s;
}

// A grid node's product with its stencil, v read through `at`.
template <class V>
__device__ __forceinline__ double stencil(const MgLevel &l, int at, V v) {
  const gptr<float> a = global_ptr(l.a);
  float c[25], x[25];
#pragma unroll
  for (int o = 0; o < 25; o++) {
    c[o] = a[(size_t)o * l.pn + at];
    x[o] = v[at + (o / 5 - 2) * l.px + o % 5 - 2];
  }
  double s = 0.0;
#pragma unroll
  for (int o = 0; o < 25; o++) s += (double)c[o] * (double)x[o];
  return s;
}

// t = b - A x on grid k
__global__ void __launch_bounds__(NT)
    gk_res(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys,
           int k) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgLevel &l = D[m.x].lv[k];
  const int id = m.y * NT + threadIdx.x;
  if (id >= l.nx * l.ny) return;
  const int at = mg_at(l.px, id % l.nx, id / l.nx);
  global_mut(l.t)[at] = (float)((double)global_ptr(l.b)[at] - stencil(l, at, global_ptr(l.x)));
}

template <class V>
__device__ __forceinline__ float restrict_at(V t, int px, int X, int Y) {
  const int at = mg_at(px, 2 * X, 2 * Y);
  return t[at] + 0.5f * ((t[at - 1] + t[at + 1]) + (t[at - px] + t[at + px])) +
         0.25f * ((t[at - px - 1] + t[at - px + 1]) + (t[at + px - 1] + t[at + px + 1]));
}

// grid k: b = P^T t of grid k - 1 and the first smoothing step from zero.
// The nodes just outside grid k - 1 are its halo, where t stays zero.
__global__ void __launch_bounds__(NT)
    gk_restrict(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
                int sys, int k) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgLevel &f = D[m.x].lv[k - 1], &l = D[m.x].lv[k];
  const int id = m.y * NT + threadIdx.x;
  if (id >= l.nx * l.ny) return;
  const int X = id % l.nx, Y = id / l.nx, at = mg_at(l.px, X, Y);
  const float s = restrict_at(global_ptr(f.t), f.px, X, Y);
  global_mut(l.b)[at] = s;
  global_mut(l.x)[at] = OM * global_ptr(l.minv)[at] * s;
}

template <class V>
__device__ __forceinline__ float prolong_at(V xc, int px, int x, int y) {
  const int at = mg_at(px, x >> 1, y >> 1), ax = x & 1, ay = y & 1;
  // the four nodes around (weights 1, 1/2 or 1/4)
  return 0.25f * ((xc[at] + xc[at + ax]) + (xc[at + ay * px] + xc[at + ay * px + ax]));
}

// t = x + P x of grid k + 1
__global__ void __launch_bounds__(NT)
    gk_prolong(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
               int sys, int k) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgLevel &l = D[m.x].lv[k], &c = D[m.x].lv[k + 1];
  const int id = m.y * NT + threadIdx.x;
  if (id >= l.nx * l.ny) return;
  const int x = id % l.nx, y = id / l.nx, at = mg_at(l.px, x, y);
  global_mut(l.t)[at] = global_ptr(l.x)[at] + prolong_at(global_ptr(c.x), c.px, x, y);
}

// x = t + w M^-1 (b - A t)
__global__ void __launch_bounds__(NT)
    gk_smooth(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
              int sys, int k) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgLevel &l = D[m.x].lv[k];
  const int id = m.y * NT + threadIdx.x;
  if (id >= l.nx * l.ny) return;
  const int at = mg_at(l.px, id % l.nx, id / l.nx);
  const gptr<float> t = global_ptr(l.t);
  const float res = (float)((double)global_ptr(l.b)[at] - stencil(l, at, t));
  global_mut(l.x)[at] = fmaf(OM * global_ptr(l.minv)[at], res, t[at]);
}

// The grids from d.tail on, in one workgroup: vectors in LDS, stencils read
// from the caches.  LDS: x, b and t of every grid of the tail.
__global__ void __launch_bounds__(RT)
    mk_tail(const MgSys *__restrict__ D, const MgScal *S, const int *__restrict__ list, int sys) {
  if (list) sys = list[blockIdx.x];
  if (S[sys].status != ST_RUN) return;
  extern __shared__ float lds[];
  const MgSys &d = D[sys];
  const int tid = threadIdx.x, first = d.tail, last = d.nlev - 1;
  int tot = 0;
  for (int k = first; k <= last; k++) tot += d.lv[k].pn;
  for (int i = tid; i < 3 * tot; i += RT) lds[i] = 0.0f;
  __syncthreads();
  // x, b, t of grid k at off(k), off(k) + tot, off(k) + 2 tot
  {
    const MgLevel &l = d.lv[first];
    for (int id = tid; id < l.nx * l.ny; id += RT) {
      const int at = mg_at(l.px, id % l.nx, id / l.nx);
      lds[at] = global_ptr(l.x)[at];
      lds[tot + at] = global_ptr(l.b)[at];
    }
  }
  __syncthreads();
  int off = 0;
  for (int k = first; k < last; k++) {  // down
    const MgLevel &l = d.lv[k], &c = d.lv[k + 1];
    float *x = lds + off, *b = x + tot, *t = b + tot;
    for (int id = tid; id < l.nx * l.ny; id += RT) {
      const int at = mg_at(l.px, id % l.nx, id / l.nx);
      t[at] = (float)((double)b[at] - stencil(l, at, x));
    }
    __syncthreads();
    float *xc = x + l.pn, *bc = xc + tot;
    for (int id = tid; id < c.nx * c.ny; id += RT) {
      const int X = id % c.nx, Y = id / c.nx, at = mg_at(c.px, X, Y);
      const float s = restrict_at(t, l.px, X, Y);
      bc[at] = s;
      xc[at] = OM * global_ptr(c.minv)[at] * s;
    }
    __syncthreads();
    off += l.pn;
  }
  {  // last grid: the dense inverse
    const MgLevel &l = d.lv[last];
    const int nn = l.nx * l.ny;
    float *x = lds + off, *b = x + tot;
    for (int i = tid; i < nn; i += RT) {
      float s = 0.0f;
      for (int j = 0; j < nn; j++)
        s = fmaf(global_ptr(d.cinv)[j * nn + i], b[mg_at(l.px, j % l.nx, j / l.nx)], s);
      x[mg_at(l.px, i % l.nx, i / l.nx)] = s;
    }
    __syncthreads();
  }
  for (int k = last - 1; k >= first; k--) {  // up
    const MgLevel &l = d.lv[k], &c = d.lv[k + 1];
    off -= l.pn;
    float *x = lds + off, *b = x + tot, *t = b + tot, *xc = x + l.pn;
    for (int id = tid; id < l.nx * l.ny; id += RT) {
      const int px = id % l.nx, py = id / l.nx, at = mg_at(l.px, px, py);
      t[at] = x[at] + prolong_at(xc, c.px, px, py);
    }
    __syncthreads();
    for (int id = tid; id < l.nx * l.ny; id += RT) {
      const int at = mg_at(l.px, id % l.nx, id / l.nx);
      const float res = (float)((double)b[at] - stencil(l, at, t));
      x[at] = fmaf(OM * global_ptr(l.minv)[at], res, t[at]);
    }
    __syncthreads();
  }
  const MgLevel &l = d.lv[first];
  for (int id = tid; id < l.nx * l.ny; id += RT) {
    const int at = mg_at(l.px, id % l.nx, id / l.nx);
    global_mut(l.x)[at] = lds[at];
  }
}

// t = x0 + sqrt(a_ii) P x of the first grid
__global__ void __launch_bounds__(NT)
    mk_prolong(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
               int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const MgLevel &l = d.lv[0];
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  float v = global_ptr(d.x0)[i];
  const int c = global_ptr(d.cell)[i];
  if (c >= 0) {
    const gptr<float> x = global_ptr(l.x);
    const f2_t f = frac_ptr(d)[i];
    const int at = mg_at(l.px, c % (l.nx - 1), c / (l.nx - 1));
    const float s = (1.0f - f.x) * (1.0f - f.y) * x[at] + f.x * (1.0f - f.y) * x[at + 1] +
                    (1.0f - f.x) * f.y * x[at + l.px] + f.x * f.y * x[at + l.px + 1];
    v = fmaf(global_ptr(d.sq)[i], s, v);
  }
  global_mut(d.t)[i] = v;
}

// z = S (t + w M^-1 (rs - Â t)); partials of r.z
__global__ void __launch_bounds__(NT)
    mk_post(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  double v[1] = {0.0};
  if (i < d.npad) {
    const gptr<float> t = global_ptr(d.t);
    const double res = (double)global_ptr(d.rs)[i] - (double)t[i] -
                       dot32(d, i, [&](int c) { return t[c]; });
    const float zi = (float)(fma((double)(OM * global_ptr(d.minv)[i]), res, (double)t[i]) *
                             global_ptr(d.dsq)[i]);
    global_mut(d.z)[i] = zi;
    v[0] = global_ptr(d.r)[i] * (double)zi;
  }
  put_partials<1>(v, d.part, d.nblk, m.y);
}

__global__ void __launch_bounds__(RT)
    ms_beta(const MgSys *__restrict__ D, MgScal *S_, const int *__restrict__ list, int sys) {
  if (list) sys = list[blockIdx.x];
  MgScal *S = S_ + sys;
  if (S->status != ST_RUN) return;
  double t[1];
  sum_partials<1>(D[sys].part, D[sys].nblk, t);
  if (threadIdx.x != 0) return;
  const double rz = t[0];
  if (rz != rz || !isfinite(rz)) S->status = ST_NAN;
  else if (!(rz > 0.0)) S->status = ST_BREAK;
  else {
    S->beta = S->first ? 0.0 : rz / S->rz;
    S->rz = rz;
    S->first = 0;
  }
}

// ------------------------------------------------------------------ the plan

// Each row's point.  Mesh systems: P1 the node (ends null), P2 the vertex or
// the edge's midpoint (ends: mesh-internal vertices).  Sparse systems whose
// rows are a mesh's dofs (perm not null): caller's row order[i] (order null:
// i), a vertex below nnode, else the edge's midpoint.
__global__ void __launch_bounds__(NT)
    plan_points(int n, const double2 *__restrict__ xy, const int2 *__restrict__ ends,
                const int *__restrict__ order, const int *__restrict__ perm, int nnode,
                const long long *__restrict__ edges, long long nedges,
                double2 *__restrict__ pt) {
  const int i = blockIdx.x * NT + threadIdx.x;
  if (i >= n) return;
  int a, b;
  if (perm) {
    const int u = order ? order[i] : i;
    if (u < nnode) {
      a = b = perm[u];
    } else {
      a = perm[edges[u - nnode] - 1];
      b = perm[edges[nedges + u - nnode] - 1];
    }
  } else if (ends) {
    a = ends[i].x;
    b = ends[i].y;
  } else {
    a = b = i;
  }
  const double2 p = xy[a], q = xy[b];
  pt[i] = make_double2(0.5 * (p.x + q.x), 0.5 * (p.y + q.y));
}

// A row takes part in the grids when it is no Dirichlet row and is coupled
// to another one.
__device__ __forceinline__ bool takes_part(int i, const int *__restrict__ row_bd,
                                           const int *__restrict__ sp,
                                           const int *__restrict__ sc) {
  if (row_bd[i] >= 0) return false;
  const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
  for (int k = 0; k < w; k++)
    if (sc[off + 64 * k] != i) return true;
  return false;
}

// Per block: the interior rows' bounding box, count and largest coupling
// extents (|dx|, |dy| over the matrix entries).
__global__ void __launch_bounds__(NT)
    plan_extent(int n, const double2 *__restrict__ pt, const int *__restrict__ row_bd, const int *__restrict__ sp,
                const int *__restrict__ sc, double *__restrict__ out) {
  const int i = blockIdx.x * NT + threadIdx.x;
  // min x, min y, -max x, -max y, -max |dx|, -max |dy|
  double v[6] = {1e300, 1e300, 1e300, 1e300, 0.0, 0.0};
  double cnt = 0.0;
  if (i < n && takes_part(i, row_bd, sp, sc)) {
    const double2 a = pt[i];
    v[0] = a.x;
    v[1] = a.y;
    v[2] = -a.x;
    v[3] = -a.y;
    cnt = 1.0;
    const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
    for (int k = 0; k < w; k++) {
      const int j = sc[off + 64 * k];
      if (j >= n) continue;
      const double2 b = pt[j];
      v[4] = fmin(v[4], -fabs(a.x - b.x));
      v[5] = fmin(v[5], -fabs(a.y - b.y));
    }
  }
  __shared__ double sh[7][NT / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < 6; j++) {
    double t = v[j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t = fmin(t, __shfl_xor(t, o, 64));
    if (lane == 0) sh[j][wv] = t;
  }
  cnt = wave_sum(cnt);
  if (lane == 0) sh[6][wv] = cnt;
  __syncthreads();
  if (threadIdx.x < 7) {
    double t = sh[threadIdx.x][0];
    for (int k = 1; k < NT / 64; k++)
      t = threadIdx.x < 6 ? fmin(t, sh[threadIdx.x][k]) : t + sh[threadIdx.x][k];
    out[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
  }
}

__global__ void __launch_bounds__(NT)
    plan_area(int nelem, const double *__restrict__ area, double *__restrict__ out) {
  double s = 0.0;
  for (int e = blockIdx.x * NT + threadIdx.x; e < nelem; e += gridDim.x * NT) s += area[e];
  __shared__ double sh[NT / 64];
  s = block_sum<NT>(s, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// Each row's cell (-1: takes no part) and its position in it; key: the cell,
// the rows that take no part last.
__global__ void __launch_bounds__(NT)
    plan_cells(int n, int npad, const double2 *__restrict__ pt, const int *__restrict__ row_bd,
               const int *__restrict__ sp, const int *__restrict__ sc, double x0, double y0, double hx, double hy,
               int ncx, int ncy, int *__restrict__ cell, float2 *__restrict__ frac,
               int *__restrict__ key, int *__restrict__ row) {
  const int i = blockIdx.x * NT + threadIdx.x;
  if (i >= npad) return;
  int c = -1;
  float2 f = make_float2(0.0f, 0.0f);
  if (i < n && takes_part(i, row_bd, sp, sc)) {
    const double2 a = pt[i];
    const double tx = (a.x - x0) / hx, ty = (a.y - y0) / hy;
    const int ix = min(max((int)floor(tx), 0), ncx - 1), iy = min(max((int)floor(ty), 0), ncy - 1);
    f = make_float2(fminf(fmaxf((float)(tx - ix), 0.0f), 1.0f),
                    fminf(fmaxf((float)(ty - iy), 0.0f), 1.0f));
    c = iy * ncx + ix;
  }
  cell[i] = c;
  frac[i] = f;
  if (i < n) {
    key[i] = c < 0 ? ncx * ncy : c;
    row[i] = i;
  }
}

// first sorted position of each cell (keys sorted; cell ncell: the end)
__global__ void __launch_bounds__(NT)
    plan_cptr(int n, int ncell, const int *__restrict__ key, int *__restrict__ cptr) {
  const int c = blockIdx.x * NT + threadIdx.x;
  if (c > ncell) return;
  int lo = 0, hi = n;  // first position with key >= c
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (key[mid] < c) lo = mid + 1;
    else hi = mid;
  }
  cptr[c] = lo;
}

// Per block: occupied cells and the most rows of one.
__global__ void __launch_bounds__(NT)
    plan_fill(int ncell, const int *__restrict__ cptr, int *__restrict__ out) {
  const int c = blockIdx.x * NT + threadIdx.x;
  int k = c < ncell ? cptr[c + 1] - cptr[c] : 0, occ = k > 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    k = max(k, __shfl_xor(k, o, 64));
    occ += __shfl_xor(occ, o, 64);
  }
  __shared__ int sh[2][NT / 64];
  if ((threadIdx.x & 63) == 0) {
    sh[0][threadIdx.x >> 6] = k;
    sh[1][threadIdx.x >> 6] = occ;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NT / 64; w++) {
      k = max(k, sh[0][w]);
      occ += sh[1][w];
    }
    out[2 * blockIdx.x] = k;
    out[2 * blockIdx.x + 1] = occ;
  }
}

// The plan of a mesh system, or of a sparse system whose rows are the dofs
// of mesh m (row i: the caller's order[i], order null: i).
MgPlan *build_plan(System &s, const Mesh &m, const int *order, hipStream_t st) {
  MgPlan *pl = new MgPlan();
  try {
    const int n = s.n, np = s.npad;
    const bool own = s.mesh != nullptr;
    const unsigned g = nb(n, NT);
    DevBuf<double> ext((size_t)7 * g), ar(256);
    DevBuf<double2> pt(n);
    plan_points<<<g, NT, 0, st>>>(n, m.xy.p, own && s.degree == 2 ? s.d_dof_ends.p : nullptr,
                                  order, own ? nullptr : m.d_perm.p, m.nnode, m.d_edges.p,
                                  m.nedges, pt.p);
    plan_extent<<<g, NT, 0, st>>>(n, pt.p, s.d_row_bd.p, s.d_slice_ptr.p, s.d_sell_col.p, ext.p);
    plan_area<<<256, NT, 0, st>>>(m.nelem, m.area.p, ar.p);
    HIPCHECK(hipGetLastError());
    std::vector<double> he((size_t)7 * g), ha(256);
    HIPCHECK(hipMemcpyAsync(he.data(), ext.p, ext.bytes(), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipMemcpyAsync(ha.data(), ar.p, ar.bytes(), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    double v[7] = {1e300, 1e300, 1e300, 1e300, 0, 0, 0}, area = 0.0;
    for (int j = 0; j < 7; j++)
      for (unsigned b = 0; b < g; b++)
        v[j] = j < 6 ? std::min(v[j], he[(size_t)j * g + b]) : v[j] + he[(size_t)j * g + b];
    for (double a : ha) area += a;
    const double lx = -v[2] - v[0], ly = -v[3] - v[1], ex = -v[4], ey = -v[5], rows = v[6];
    if (!(rows > 0 && area > 0 && std::isfinite(area) && lx > 0 && ly > 0 && ex > 0 && ey > 0))
      return pl;
    // cells of four rows' area in the couplings' aspect, and at least the
    // couplings' extents (then a coupling stays within neighbouring cells,
    // which keeps the first grid's stencil at 25 points)
    const double c = std::sqrt(4.0 * area / rows / (ex * ey));
    const double hx = ex * std::max(c, 1.0001), hy = ey * std::max(c, 1.0001);
    const double x0 = v[0] - 0.25 * hx, y0 = v[1] - 0.25 * hy;
    const double fx = (lx + 0.25 * hx) / hx, fy = (ly + 0.25 * hy) / hy;
    if (!(fx < 1e6 && fy < 1e6)) return pl;
    int nx = (int)std::floor(fx) + 2, ny = (int)std::floor(fy) + 2;
    if ((double)nx * ny > 0.75 * rows) return pl;
    const int ncx = nx - 1, ncy = ny - 1, ncell = ncx * ncy;
    DevBuf<int> key(n), row(n), skey(n), fill(2 * nb(ncell, NT));
    pl->cell.alloc(np);
    pl->frac.alloc(np);
    pl->crow.alloc(n);
    pl->cptr.alloc(ncell + 1);
    plan_cells<<<nb(np, NT), NT, 0, st>>>(n, np, pt.p, s.d_row_bd.p, s.d_slice_ptr.p,
                                          s.d_sell_col.p, x0, y0, hx, hy, ncx, ncy, pl->cell.p, pl->frac.p, key.p, row.p);
    HIPCHECK(hipGetLastError());
    int bits = 1;
    while (ncell >> bits) bits++;
    size_t tmp = 0;
    HIPCHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, key.p, skey.p, row.p, pl->crow.p, n,
                                                0, bits, st));
    DevBuf<char> t(std::max<size_t>(tmp, 1));
    HIPCHECK(hipcub::DeviceRadixSort::SortPairs(t.p, tmp, key.p, skey.p, row.p, pl->crow.p, n, 0,
                                                bits, st));
    plan_cptr<<<nb(ncell + 1, NT), NT, 0, st>>>(n, ncell, skey.p, pl->cptr.p);
    plan_fill<<<nb(ncell, NT), NT, 0, st>>>(ncell, pl->cptr.p, fill.p);
    HIPCHECK(hipGetLastError());
    std::vector<int> hf(fill.n);
    HIPCHECK(hipMemcpyAsync(hf.data(), fill.p, fill.bytes(), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    int most = 0;
    double occ = 0;
    for (size_t k = 0; k < hf.size(); k += 2) {
      most = std::max(most, hf[k]);
      occ += hf[k + 1];
    }
    // a graded mesh puts many rows into some cells: the grid is then too
    // coarse there for the smoother, and plain Jacobi-PCG keeps the system
    if (rows > 10.0 * occ || most > 64) return pl;
    int k = 0;
    pl->tail = -1;
    for (;; k++) {
      if (k == MG_MAXLEV) return pl;
      pl->nx[k] = nx;
      pl->ny[k] = ny;
      pl->px[k] = nx + 2 * MG_HALO;
      pl->pn[k] = (pl->px[k] * (ny + 2 * MG_HALO) + 63) / 64 * 64;
      if (pl->tail < 0 && pl->pn[k] <= MG_TAIL) pl->tail = k;
      if (nx * ny <= MG_DENSE) break;
      nx = nx / 2 + 1;
      ny = ny / 2 + 1;
    }
    pl->nlev = k + 1;
    if (pl->tail < 0) return pl;
    pl->ok = true;
    return pl;
  } catch (...) {
    delete pl;
    throw;
  }
}

size_t tail_lds(const MgPlan &pl) {
  size_t t = 0;
  for (int k = pl.tail; k < pl.nlev; k++) t += pl.pn[k];
  return 3 * t * sizeof(float);
}

}  // namespace

void mg_plan_free(MgPlan *p) { delete p; }

const MgPlan *mg_plan(System &s, hipStream_t st) {
  if (!s.mg_plan && s.mesh) s.mg_plan = build_plan(s, *s.mesh, nullptr, st);
  return s.mg_plan && s.mg_plan->ok ? s.mg_plan : nullptr;
}

size_t mg_grid_floats(const MgPlan &pl) {
  size_t f = 0;
  for (int k = 0; k < pl.nlev; k++) f += (size_t)29 * pl.pn[k];
  return f + MG_DENSE * MG_DENSE;
}

void mg_grid_layout(const MgPlan &pl, float *base, MgSys &d) {
  d.cell = pl.cell.p;
  d.frac = pl.frac.p;
  d.cptr = pl.cptr.p;
  d.crow = pl.crow.p;
  d.nlev = pl.nlev;
  d.tail = pl.tail;
  for (int k = 0; k < pl.nlev; k++) {
    MgLevel &l = d.lv[k];
    const size_t pn = pl.pn[k];
    l.nx = pl.nx[k];
    l.ny = pl.ny[k];
    l.px = pl.px[k];
    l.pn = (int)pn;
    l.a = base;
    l.minv = base + 25 * pn;
    l.x = l.minv + pn;
    l.b = l.x + pn;
    l.t = l.b + pn;
    base += 29 * pn;
  }
  d.cinv = base;
}

struct MgWork {
  MgSys h{};                     // the descriptor (host copy)
  DevBuf<MgSys> d;
  DevBuf<MgScal> sc;
  MgScal *h_sc = nullptr;        // pinned
  DevBuf<double> x, r, q, p0, p1, dsq, part;
  DevBuf<float> sv32, sq, minv, z, rs, x0, t, grid;
  int nblk = 0;
  uint64_t version = 0;          // of the matrix the set-up was made from
  uint64_t rowsum_version = 0;   // of the matrix the row sums were taken of
  double rowsum = 0.0;
  hipStream_t cap = nullptr;
  hipGraphExec_t graph = nullptr;
  ~MgWork() {
    if (graph) (void)hipGraphExecDestroy(graph);
    if (cap) (void)hipStreamDestroy(cap);
    if (h_sc) (void)hipHostFree(h_sc);
  }
};

void mg_work_free(MgWork *w) { delete w; }

namespace {

MgWork *ensure_work(System &s, const MgPlan &pl, hipStream_t st) {
  if (s.mg_work) return s.mg_work;
  MgWork *w = new MgWork();
  try {
    const size_t np = s.npad;
    w->nblk = (int)(nb(np, NT) + 7) / 8 * 8;  // a multiple of 8: the XCD deal
    w->x.alloc(np);
    w->r.alloc(np);
    w->q.alloc(np);
    w->p0.alloc(np);
    w->p1.alloc(np);
    w->dsq.alloc(np);
    w->part.alloc((size_t)4 * w->nblk + 1);
    w->sv32.alloc(std::max(1, s.slice_ptr.back()));
    w->sq.alloc(np);
    w->minv.alloc(np);
    w->z.alloc(np);
    w->rs.alloc(np);
    w->x0.alloc(np);
    w->t.alloc(np);
    w->grid.alloc(mg_grid_floats(pl));
    w->d.alloc(1);
    w->sc.alloc(1);
    HIPCHECK(hipHostMalloc((void **)&w->h_sc, sizeof(MgScal), hipHostMallocDefault));
    MgSys &d = w->h;
    d.sp = s.d_slice_ptr.p;
    d.sc = s.d_sell_col.p;
    d.sd = s.d_sell_d16.p;
    d.row_bd = s.d_row_bd.p;
    d.sv64 = s.d_sell_val.p;
    d.diag = s.d_diag.p;
    d.sv32 = w->sv32.p;
    d.dsq = w->dsq.p;
    d.sq = w->sq.p;
    d.minv = w->minv.p;
    d.x = w->x.p;
    d.r = w->r.p;
    d.q = w->q.p;
    d.p[0] = w->p0.p;
    d.p[1] = w->p1.p;
    d.z = w->z.p;
    d.rs = w->rs.p;
    d.x0 = w->x0.p;
    d.t = w->t.p;
    d.part = w->part.p;
    d.n = s.n;
    d.npad = s.npad;
    d.nblk = w->nblk;
    mg_grid_layout(pl, w->grid.p, d);
    mk_zero<<<nb(w->grid.n, 256), 256, 0, st>>>(w->grid.p, w->grid.n);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipMemcpyAsync(w->d.p, &d, sizeof(MgSys), hipMemcpyHostToDevice, st));
    HIPCHECK(hipStreamSynchronize(st));
  } catch (...) {
    delete w;
    throw;
  }
  s.mg_work = w;
  return w;
}

}  // namespace

// The set-up of one matrix (descriptor `sys` of D): fine scaling, the grids'
// matrices and smoothing weights, the last grid's inverse.
void mg_setup(const MgPlan &pl, int nblk, const MgSys *D, int sys, hipStream_t st) {
  mk_scale<<<nblk, NT, 0, st>>>(nullptr, D, sys);
  mk_galerkin<<<nb(pl.nx[0] * pl.ny[0], GT), GT, 0, st>>>(nullptr, D, sys);
  for (int k = 0; k < pl.tail; k++) {
    gk_weights<<<nb(pl.nx[k] * pl.ny[k], GT), GT, 0, st>>>(nullptr, D, sys, k);
    gk_galerkin<<<nb(pl.nx[k + 1] * pl.ny[k + 1], GT), GT, 0, st>>>(nullptr, D, sys, k + 1);
  }
  mk_tail_setup<<<1, ST, 0, st>>>(D, nullptr, sys);
  HIPCHECK(hipGetLastError());
}

namespace {

void v_cycle(const MgPlan &pl, MgWork *w, hipStream_t st) {
  const MgSys *D = w->d.p;
  MgScal *S = w->sc.p;
  auto grid = [&](int k) { return nb(pl.nx[k] * pl.ny[k], NT); };
  mk_res<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  mk_restrict<<<grid(0), NT, 0, st>>>(nullptr, D, S, 0);
  for (int k = 0; k < pl.tail; k++) {
    gk_res<<<grid(k), NT, 0, st>>>(nullptr, D, S, 0, k);
    gk_restrict<<<grid(k + 1), NT, 0, st>>>(nullptr, D, S, 0, k + 1);
  }
  mk_tail<<<1, RT, tail_lds(pl), st>>>(D, S, nullptr, 0);
  for (int k = pl.tail - 1; k >= 0; k--) {
    gk_prolong<<<grid(k), NT, 0, st>>>(nullptr, D, S, 0, k);
    gk_smooth<<<grid(k), NT, 0, st>>>(nullptr, D, S, 0, k);
  }
  mk_prolong<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  mk_post<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  ms_beta<<<1, RT, 0, st>>>(D, S, nullptr, 0);
}

void iteration(const MgPlan &pl, MgWork *w, hipStream_t st) {
  const MgSys *D = w->d.p;
  MgScal *S = w->sc.p;
  mk_dir<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  ms_alpha<<<1, RT, 0, st>>>(D, S, nullptr, 0);
  mk_update<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  v_cycle(pl, w, st);
}

// Whether the V-cycle pays for the assembled matrix: not when a mass term
// dominates it.  Jacobi-PCG's condition number is about 2 over the smallest
// row sum over diagonal (1 for a lumped mass matrix, O(h^2) for a stiffness
// matrix); at 0.2 it needs about as many launches as the V-cycles do.
constexpr double MASS_DOMINANT = 0.2;
bool mg_pays(System &s, MgWork *w, hipStream_t st) {
  if (!s.mass) return true;
  if (w->rowsum_version != s.a_version) {
    const unsigned g = nb(s.n, NT);
    mk_rowsum<<<g, NT, 0, st>>>(s.n, s.d_row_bd.p, s.d_slice_ptr.p, s.d_sell_val.p, s.d_diag.p,
                                w->part.p);
    ms_rowsum<<<1, RT, 0, st>>>((int)g, w->part.p);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipMemcpyAsync(&w->rowsum, w->part.p, sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    w->rowsum_version = s.a_version;
  }
  return !(w->rowsum > MASS_DOMINANT);
}

constexpr int GRAPH_ITERS = 2;

// GRAPH_ITERS iterations, captured once per system (every pointer comes from
// the device descriptor) and replayed.
void launch_graph(const MgPlan &pl, MgWork *w, hipStream_t st) {
  if (!w->graph) {
    if (!w->cap) HIPCHECK(hipStreamCreateWithFlags(&w->cap, hipStreamNonBlocking));
    hipGraph_t g;
    HIPCHECK(hipStreamBeginCapture(w->cap, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < GRAPH_ITERS; k++) iteration(pl, w, w->cap);
    HIPCHECK(hipStreamEndCapture(w->cap, &g));
    hipGraphExec_t ex;
    const hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    HIPCHECK(e);
    w->graph = ex;
  }
  HIPCHECK(hipGraphLaunch(w->graph, st));
}

}  // namespace

// Systems below this many rows stay with Jacobi-PCG.
constexpr int MG_MIN_ROWS = 4096;

// A sparse system's rows are the dofs of mesh m (m null: unknown, and it is
// Jacobi-PCG's); its plan is kept for as long as the mesh stays the same one.
void mg_set_mesh(System &s, const Mesh *m, const int *order, hipStream_t st) {
  s.mg_off = !m || m->ndof != s.n || s.n < MG_MIN_ROWS;
  if (s.mg_off || (s.mg_plan && s.mg_serial == m->serial)) return;
  if (s.mg_work) mg_work_free(s.mg_work);
  if (s.mg_plan) mg_plan_free(s.mg_plan);
  s.mg_work = nullptr;
  s.mg_plan = nullptr;
  s.mg_plan = build_plan(s, *m, order, st);
  s.mg_serial = m->serial;
  s.mass = true;  // the matrix is the caller's: look before using the grids
}

// Solves by multigrid CG when that suits the system; false when it is
// Jacobi-PCG's.
bool mg_solve(System &s, const double *b, double *x_out, const admfem_solve_opts &o,
              admfem_solve_stats &stats, hipStream_t st) {
  if (s.mg_off || s.n < MG_MIN_ROWS) return false;
  auto t0 = std::chrono::steady_clock::now();
  const MgPlan *plan = mg_plan(s, st);
  if (!plan) return false;
  const MgPlan &pl = *plan;
  MgWork *w = ensure_work(s, pl, st);
  if (!mg_pays(s, w, st)) return false;
  const MgSys *D = w->d.p;
  MgScal *S = w->sc.p;
  if (w->version != s.a_version) {  // a new matrix
    mg_setup(pl, w->nblk, D, 0, st);
    w->version = s.a_version;
  }
  mk_start<true><<<w->nblk, NT, 0, st>>>(nullptr, D, 0, b);
  ms_start<<<1, RT, 0, st>>>(D, S, 0, 1, o.rtol * o.rtol, o.max_iter);
  int it = 0;
  double true_prev = -1.0, rr_true = 0.0;
  for (int restarts = 0;; restarts++) {
    v_cycle(pl, w, st);
    int chunk = o.check_every > 0 ? o.check_every : restarts ? 2 : 10;
    for (;;) {
      const int stop = (int)std::min<int64_t>((int64_t)it + chunk, o.max_iter);
      while (it < stop) {
        if (o.check_every != 1 && it + GRAPH_ITERS <= stop) {
          launch_graph(pl, w, st);
          it += GRAPH_ITERS;
        } else {
          iteration(pl, w, st);
          it++;
        }
      }
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipMemcpyAsync(w->h_sc, S, sizeof(MgScal), hipMemcpyDeviceToHost, st));
      HIPCHECK(hipStreamSynchronize(st));
      if (w->h_sc->status != ST_RUN || it >= o.max_iter) break;
      if (o.check_every <= 0) chunk = 2;
    }
    const int status = w->h_sc->status;
    it = w->h_sc->it;
    // the residual of the returned x, from the FP64 matrix
    mk_start<false><<<w->nblk, NT, 0, st>>>(nullptr, D, 0, b);
    ms_start<<<1, RT, 0, st>>>(D, S, 0, 0, 0.0, 0);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipMemcpyAsync(w->h_sc, S, sizeof(MgScal), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    rr_true = w->h_sc->rr;
    w->h_sc->status = status;
    // the recursive residual decides only when the true one agrees;
    // otherwise CG restarts from the true one, until that no longer helps
    if (status != ST_CONV || rr_true <= w->h_sc->tol2 || it >= o.max_iter || restarts >= 8 ||
        (true_prev >= 0.0 && !(rr_true < 0.25 * true_prev)))
      break;
    true_prev = rr_true;
  }
  HIPCHECK(hipMemcpyAsync(x_out, w->x.p, sizeof(double) * s.n, hipMemcpyDeviceToDevice, st));
  HIPCHECK(hipStreamSynchronize(st));
  const MgScal &h = *w->h_sc;
  stats.iterations = h.it;
  stats.replacements = h.nrepl - 1;
  stats.rel_residual = h.bb > 0 ? std::sqrt(rr_true / h.bb) : 0.0;
  switch (h.status) {
    case ST_CONV: stats.status = ADMFEM_OK; break;
    case ST_NAN: stats.status = ADMFEM_ERR_NAN; break;
    case ST_BREAK: stats.status = ADMFEM_ERR_BREAKDOWN; break;
    default: stats.status = ADMFEM_ERR_NOT_CONVERGED; break;
  }
  stats.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return true;
}

}  // namespace admfem
