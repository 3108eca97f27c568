// Multigrid-preconditioned conjugate gradients for the systems of meshes:
// FP64 CG on the Dirichlet-eliminated matrix, its preconditioner one V-cycle
// over a hierarchy of uniform grids.
//
// Jacobi-PCG takes O(1/h) iterations (4,800 at 1024^2); the V-cycle keeps the
// count at 11 - 13 for P1 at every size (P2: 12 - 15), so a solve reads the
// matrix about 60 times in all.  One forward + adjoint on MI355X, Jacobi-PCG
// -> this: Poisson 64^2 FP64 9.0 -> 1.0 ms, 511^2 FP64 79 -> 2.3 ms, 1024^2
// mixed 265 -> 4.5 ms, heat 200^2 15.6 -> 1.4 ms, P2 101^2 40 -> 2.1 ms; the
// small ones are bound by launches that depend on each other (4 - 5 us each,
// the tail 12 - 15), the large ones by the fine level's passes over memory.
//
// The grids are laid over the mesh's bounding box (cells of about four rows)
// and know nothing of the triangles: a row takes part through the bilinear
// interpolation P from the four nodes of its cell, and every coarse matrix is
// the Galerkin product P^T A P of the assembled matrix, a 25-point stencil on
// each grid, so boundary conditions, holes, coefficients and mass terms need no
// special case.  Rows of Dirichlet nodes are not interpolated.
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
// FP32's range is no limit on A or b: the V-cycle sees s^2 A and sc r, with s
// from the diagonal (matrix_unit) and sc from the first residual (ms_start),
// and mk_dir takes z back by s^2 / sc.  Both are powers of two, so the
// mantissas, and with them the iterates, are those of the unscaled numbers.
// A solve is converged when the residual recomputed from the FP64 matrix is, or
// when restarts from that residual no longer lower it: FP64's floor (ms_check).
//
// One iteration (every kernel returns at once when its system is done), from
// the fine residual after the first smoothing step (mk_step; mk_lead when CG
// starts):
//   mk_res       residual after the second one; plans with two steps
//   mk_restrict  to the first grid, with its first smoothing step
//   gk_down      the grids down to MG_TAIL nodes: residual and restriction of
//                a tile in one launch
//   mk_tail      the remaining grids, one workgroup per system, in LDS
//   gk_up        and up: prolongation and smoothing of a tile; the first grid
//                also interpolates its rows
//   mk_mid, mk_post  the fine level's smoothing (mk_mid: plans with two
//                steps): z, partials of r.z
//   mk_dir       beta = r.z / previous r.z, p = z + beta p, q = A p; partials
//                of p.q, r.q, q.q, r.r
//   mk_step      alpha = r.z / p.q, the new |r|^2 = r.r - 2 alpha r.q +
//                alpha^2 q.q, x += alpha p, r -= alpha q, first smoothing step
//                and the residual after it (two steps: the second step)
// When every grid fits the tail, mk_tail also restricts and interpolates: four
// launches an iteration.  The scalars need no launch of their own: every
// block of mk_dir and mk_step sums the partials itself, in one order, and
// block 0 keeps the result for the next kernel (two copies of the state, each
// kernel reading one and writing the other).  Above MG_SUM partials one
// block sums them first (ms_reduce): 1,032 blocks reading 1,032 x 4 partials
// cost less than a launch, 4,104 blocks reading 4,104 would not.
// No atomics, no fences; every reduction has one order.
#include <hipcub/hipcub.hpp>

#include <chrono>
#include <climits>
#include <cmath>
#include <mutex>

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
// Two smoothing steps on the fine level instead (plans with steps = 2): the
// degree-2 Chebyshev polynomial of M^-1 A for its spectrum's part [1/8, 1],
// first step x + C0 M^-1 r, second x' + CM (x' - x) + C1 M^-1 r'.
constexpr float C0 = 16.0f / 9.0f, CM = 0.43369f, C1 = 2.54902f;
// Partials that the wide kernels' blocks sum themselves, at most.
constexpr int MG_SUM = 1280;

inline unsigned nb(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// The system and block of a grid block: from the batch's map, or (no map)
// system `sys` with the blocks dealt to the 8 XCDs in contiguous eighths.
__device__ __forceinline__ int2 where(const int2 *map, int sys) {
  if (map) return map[blockIdx.x];
  return make_int2(sys, xcd_block(blockIdx.x, gridDim.x));
}

typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ gptr<f2_t> frac_ptr(const float2 *p) {
  return (gptr<f2_t>)reinterpret_cast<const f2_t *>(p);
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

// A wide kernel's block's sums of NV arrays of G values (the same in every
// block); G = 1: already summed.
template <int NV>
__device__ __forceinline__ void sum_small(const double *v_, int G, double (&out)[NV]) {
  const gptr<double> v = global_ptr(v_);
  if (G == 1) {
#pragma unroll
    for (int j = 0; j < NV; j++) out[j] = v[j];
    return;
  }
  __shared__ double sh[NV][NT / 64];
  double a[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) a[j] = 0.0;
  int k = threadIdx.x;
  for (; k + 3 * NT < G; k += 4 * NT) {
    double t[NV][4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < NV; j++) t[j][u] = v[(size_t)j * G + k + u * NT];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < NV; j++) a[j] += t[j][u];
  }
  for (; k < G; k += NT)
#pragma unroll
    for (int j = 0; j < NV; j++) a[j] += v[(size_t)j * G + k];
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
    for (int w = 0; w < NT / 64; w++) t += sh[j][w];
    out[j] = t;
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

// The power of two s with s sqrt(a_ii) in [1, 2) for the largest of 64 diagonal
// entries, of rows spread evenly over the cells (by one wave: a row a lane, which
// every wave reads anew rather than wait for another launch).
__device__ __forceinline__ double matrix_unit(const MgSys &d) {
  const gptr<int> cptr = global_ptr(d.cptr), crow = global_ptr(d.crow);
  const int rows = cptr[(d.lv[0].nx - 1) * (d.lv[0].ny - 1)];
  double v = global_ptr(d.diag)[crow[(int)((int64_t)(threadIdx.x & 63) * rows >> 6)]];
  if (!(v > 0.0 && isfinite(v))) v = 0.0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v > 0.0 ? ldexp(1.0, -(ilogb(v) >> 1)) : 1.0;
}

// dsq = 1/(s sqrt(a_ii)), sq = s sqrt(a_ii), the FP32 scaled off-diagonals and
// the smoother's weights.  A row without a positive diagonal (an isolated node,
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
  const double aii = dg[i], s = matrix_unit(d);
  const double si = aii > 0.0 ? 1.0 / sqrt(aii) : 0.0;
  if (m.y == 0 && threadIdx.x == 0) *global_mut(d.unit) = s;
  global_mut(d.dsq)[i] = si / s;
  global_mut(d.sq)[i] = aii > 0.0 ? (float)(sqrt(aii) * s) : 0.0f;
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

// The first grid's matrix s^2 P^T A P: 4 GR threads per grid node, GR for each of
// its cells, which share the cell's rows; a thread's sums for the 4 x 4 nodes
// around its cell live in LDS (they are addressed by the columns' cells).
// Bound by the latency of the row -> column -> cell loads: with four lanes to a
// cell 33 -> 15 us for the 1,156 nodes of P1 64^2 and 115 -> 47 for P2 101^2.
// Past GALERKIN_SPLIT nodes (and in batches) the threads fill the chip with one
// lane each, and the LDS of the sums bounds their waves: 66,000 nodes of P1 1024^2 237
// -> 201 us (16 sums a thread instead of 25), 331 with four lanes.
constexpr int GT = 256;
constexpr int GALERKIN_SPLIT = 20000;
constexpr int mg_gn(int gr) { return GT / (4 * gr); }  // nodes of a block
template <int GR>
__global__ void __launch_bounds__(GT)
    mk_galerkin(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys) {
  constexpr int GN = mg_gn(GR);
  __shared__ double acc[16][GT];
  const int2 mb = where(map, sys);
  if (mb.x < 0) return;
  const MgSys &d = D[mb.x];
  const MgLevel &l = d.lv[0];
  const int tid = threadIdx.x, id = mb.y * GN + tid / (4 * GR), nn = l.nx * l.ny;
  const int X = id % l.nx, Y = id / l.nx, ncx = l.nx - 1, ncy = l.ny - 1;
#pragma unroll
  for (int o = 0; o < 16; o++) acc[o][tid] = 0.0;
  const int cx = X - (tid & 1), cy = Y - ((tid >> 1) & 1);
  if (id < nn && cx >= 0 && cx < ncx && cy >= 0 && cy < ncy) {
    const gptr<int> cptr = global_ptr(d.cptr), crow = global_ptr(d.crow),
                    cell = global_ptr(d.cell);
    const gptr<int> sc = global_ptr(d.sc), sp = global_ptr(d.sp);
    const gptr<double> sv = global_ptr(d.sv64), dg = global_ptr(d.diag);
    const gptr<f2_t> frac = frac_ptr(d.frac);
    const int c = cy * ncx + cx, k1 = cptr[c + 1];
    for (int k = cptr[c] + ((tid >> 2) & (GR - 1)); k < k1; k += GR) {
      const int i = crow[k];
      const f2_t f = frac[i];
      const double wi =
          (double)(cx == X ? 1.0f - f.x : f.x) * (double)(cy == Y ? 1.0f - f.y : f.y);
      const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
#pragma unroll 4
      for (int e = -1; e < w; e++) {
        const int j = e < 0 ? i : sc[off + 64 * e];
        const double v = wi * (e < 0 ? dg[i] : sv[off + 64 * e]);
        const int cj = cell[j];
        const f2_t g = frac[j];
        const int jy = cj / ncx, ox = cj - jy * ncx - cx + 1, oy = jy - cy + 1;
        // (cj < 0: no part; the plan excludes cells further off)
        if (cj < 0 || ox < 0 || ox > 2 || oy < 0 || oy > 2) continue;
        acc[oy * 4 + ox][tid] += v * ((1.0 - g.x) * (1.0 - g.y));
        acc[oy * 4 + ox + 1][tid] += v * ((double)g.x * (1.0 - g.y));
        acc[oy * 4 + ox + 4][tid] += v * ((1.0 - g.x) * (double)g.y);
        acc[oy * 4 + ox + 5][tid] += v * ((double)g.x * (double)g.y);
      }
    }
  }
  const double s = *global_ptr(d.unit), s2 = s * s;
  __syncthreads();
  for (int t = tid; t < 25 * GN; t += GT) {
    const int o = t / GN, q = t % GN, node = mb.y * GN + q;
    if (node >= nn) continue;
    double sum = 0.0;
#pragma unroll
    for (int cl = 0; cl < 4; cl++) {  // the node is (1 - (cl & 1), 1 - (cl >> 1)) of the cell's
      const int ox = o % 5 - 1 + (cl & 1), oy = o / 5 - 1 + (cl >> 1);
      if (ox < 0 || ox > 3 || oy < 0 || oy > 3) continue;
#pragma unroll
      for (int r = 0; r < GR; r++) sum += acc[oy * 4 + ox][q * 4 * GR + 4 * r + cl];
    }
    global_mut(l.a)[(size_t)o * l.pn + mg_at(l.px, node % l.nx, node / l.nx)] =
        (float)(sum * s2);
  }
}

// One node's entries of the next grid's matrix, P^T A P with the bilinear
// interpolation of a grid from every second node: the part of the finer row
// 2 Y + dy, dy in -1 .. 1 (else nothing).  a(o, x, y): the finer grid's entries.
template <class A>
__device__ __forceinline__ void coarse_part(A a, int nx, int ny, int X, int Y, int dy,
                                            double (&s)[25]) {
  double T[5][7];
#pragma unroll
  for (int u = 0; u < 5; u++)
#pragma unroll
    for (int v = 0; v < 7; v++) T[u][v] = 0.0;
  const int y = 2 * Y + dy;
  if (dy <= 1 && y >= 0 && y < ny) {
#pragma unroll
    for (int dx = -1; dx <= 1; dx++) {
      const int x = 2 * X + dx;
      if (x < 0 || x >= nx) continue;
      const double w = (dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0);
#pragma unroll
      for (int oy = 0; oy < 5; oy++)
#pragma unroll
        for (int ox = 0; ox < 5; ox++) T[oy][dx + ox + 1] += w * (double)a(oy * 5 + ox, x, y);
    }
  }
#pragma unroll
  for (int o = 0; o < 25; o++) s[o] = 0.0;
#pragma unroll
  for (int oy = 0; oy < 5; oy++) {
    double U[5];
#pragma unroll
    for (int ox = 0; ox < 5; ox++) {
      // column 2 (ox - 2) + u + 3 of T, weights 1/2, 1, 1/2
      U[ox] = 0.0;
#pragma unroll
      for (int u = -1; u <= 1; u++) {
        const int tx = 2 * ox - 1 + u;
        if (tx >= 0 && tx < 7) U[ox] += (u ? 0.5 : 1.0) * T[oy][tx];
      }
    }
#pragma unroll
    for (int cy = 0; cy < 5; cy++) {
      // finer offset dy + oy - 2 against the coarser 2 (cy - 2)
      const int v = dy + oy + 2 - 2 * cy;
      const double w = v == 0 ? 1.0 : v == 1 || v == -1 ? 0.5 : 0.0;
#pragma unroll
      for (int ox = 0; ox < 5; ox++) s[cy * 5 + ox] += w * U[ox];
    }
  }
}

// The same by the four lanes of a quad (one finer row each, one idle); put(o,
// v) stores, a quarter of the entries by each lane.
template <class A, class P>
__device__ __forceinline__ void coarse_node(A a, int nx, int ny, int X, int Y, P put) {
  const int q = threadIdx.x & 3;
  double s[25];
  coarse_part(a, nx, ny, X, Y, q - 1, s);
#pragma unroll
  for (int o = 0; o < 25; o++) {
    s[o] += __shfl_xor(s[o], 1, 64);
    s[o] += __shfl_xor(s[o], 2, 64);
    if ((o & 3) == q) put(o, (float)s[o]);
  }
}

// A grid's smoothing weight at a node.
template <class A>
__device__ __forceinline__ float weight_node(A a, int nx, int ny, int x, int y) {
  float v[25], ajj[25];
#pragma unroll
  for (int o = 0; o < 25; o++) {
    const int X = x + o % 5 - 2, Y = y + o / 5 - 2;
    v[o] = a(o, x, y);
    ajj[o] = X >= 0 && X < nx && Y >= 0 && Y < ny ? a(12, X, Y) : 0.0f;
  }
  float s = 0.0f;
#pragma unroll
  for (int o = 0; o < 25; o++)
    if (ajj[o] > 1e-30f) s += fabsf(v[o]) * rsqrtf(ajj[o]);
  return ajj[12] > 1e-30f ? rsqrtf(ajj[12]) / s : 0.0f;
}

// Grid k's weights and the matrix of grid k + 1; for the tail's first grid
// both in the form mk_tail reads them (mg.h).  Four threads a node of grid
// k + 1 (a thread's 225 dependent sums took 21 us a grid on average at P1
// 1024^2; four quarter them, 12 us), and their threads take the nodes of grid k
// in turn.
constexpr int GS = 128;
__global__ void __launch_bounds__(GS)
    gk_setup(const int2 *__restrict__ map, const MgSys *__restrict__ D, int sys, int k) {
  const int2 mb = where(map, sys);
  if (mb.x < 0) return;
  const MgSys &d = D[mb.x];
  const MgLevel &f = d.lv[k];
  const gptr<float> fa = global_ptr(f.a);
  const int px = f.px, pn = f.pn;
  auto a = [=](int o, int x, int y) { return fa[(size_t)o * pn + mg_at(px, x, y)]; };
  const int id = mb.y * GS + threadIdx.x, nf = f.nx * f.ny;
  const bool tail = k == d.tail;
  if (id < nf) {
    const int x = id % f.nx, y = id / f.nx;
    const float w = weight_node(a, f.nx, f.ny, x, y);
    global_mut(f.minv)[mg_at(px, x, y)] = w;
    if (tail) {
      float v[28];
#pragma unroll
      for (int o = 0; o < 25; o++) v[o] = a(o, x, y);
      v[25] = OM * w;
      v[26] = v[27] = 0.0f;
#pragma unroll
      for (int u = 0; u < 7; u++)
        ((gmptr<f4_t>)reinterpret_cast<f4_t *>(d.pack))[u * nf + id] =
            f4_t{v[4 * u], v[4 * u + 1], v[4 * u + 2], v[4 * u + 3]};
    }
  }
  if (k + 1 == d.nlev) return;  // (the tail's only grid)
  const MgLevel &c = d.lv[k + 1];
  const int nc = c.nx * c.ny, cid = id >> 2;
  if (cid >= nc) return;  // (whole quads)
  float *out = tail ? d.pack + 28 * nf + cid : c.a + mg_at(c.px, cid % c.nx, cid / c.nx);
  const int step = tail ? nc : c.pn;
  coarse_node(a, f.nx, f.ny, cid % c.nx, cid / c.nx,
              [&](int o, float v) { global_mut(out)[(size_t)o * step] = v; });
}

// The tail's grids below its first two, their weights and the dense inverse
// of the last one, by Gauss-Jordan on its scaled form, two pivots a barrier; a
// node whose pivot vanishes (outside the mesh, or the constant of a singular
// matrix) is left out.  The matrices live in LDS as mk_tail keeps them: a chain of
// barriers in one workgroup, bound by latency alone.
constexpr int ST = 512;
__global__ void __launch_bounds__(ST)
    mk_tail_setup(const MgSys *__restrict__ D, const int *__restrict__ list, int sys) {
  if (list) sys = list[blockIdx.x];
  if (sys < 0) return;
  const MgSys &d = D[sys];
  extern __shared__ __align__(16) float lds[];  // [25][nodes] entries and [nodes] weights a grid
  __shared__ double A[2][MG_DENSE][MG_DENSE + 1], sc[MG_DENSE];
  const int tid = threadIdx.x, last = d.nlev - 1;
  int nx = d.lv[d.tail].nx, ny = d.lv[d.tail].ny;
  float *const pack = d.pack + 28 * nx * ny;
  if (d.tail < last) {
    nx = mg_next(nx);
    ny = mg_next(ny);
    const int n0 = 25 * nx * ny;
    for (int i = tid; i < n0; i += 8 * ST) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = global_ptr(pack)[min(i + u * ST, n0 - 1)];
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (i + u * ST < n0) lds[i + u * ST] = v[u];
    }
  } else {  // one grid: its entries from the quads
    const int nn = nx * ny;
    for (int i = tid; i < 25 * nn; i += ST)
      lds[i] = global_ptr(d.pack)[((i / nn >> 2) * nn + i % nn) * 4 + (i / nn & 3)];
  }
  __syncthreads();
  float *l = lds;
  for (int k = d.tail + 1; k <= last; k++) {
    const int nn = nx * ny;
    const float *la = l;
    auto a = [=](int o, int x, int y) { return la[o * nn + y * nx + x]; };
    for (int id = tid; id < nn; id += ST)
      l[25 * nn + id] = OM * weight_node(a, nx, ny, id % nx, id / nx);
    if (k < last) {
      const int mx = mg_next(nx), my = mg_next(ny), mm = mx * my;
      float *c = l + 26 * nn;
      for (int t = tid; t < 4 * mm; t += ST) {
        const int id = t >> 2;
        coarse_node(a, nx, ny, id % mx, id / mx, [&](int o, float v) { c[o * mm + id] = v; });
      }
      l = c;
      nx = mx;
      ny = my;
    }
    __syncthreads();
  }
  const int nn = nx * ny;
  for (int i = tid; i < nn; i += ST) {
    const float aii = l[12 * nn + i];
    sc[i] = aii > 1e-30f ? 1.0 / sqrt((double)aii) : 0.0;
  }
  __syncthreads();
  for (int t = tid; t < nn * nn; t += ST) {
    const int i = t / nn, j = t % nn;
    const int dx = j % nx - i % nx, dy = j / nx - i / nx;
    double v = 0.0;
    if (abs(dx) <= 2 && abs(dy) <= 2) v = (double)l[((dy + 2) * 5 + dx + 2) * nn + i];
    A[0][i][j] = v * sc[i] * sc[j];
  }
  // (the grids' entries and weights are final: out they go meanwhile)
  if (d.tail < last) {
    const int np = (int)(l - lds) + 26 * nn;
    for (int i = tid; i < np; i += ST) global_mut(pack)[i] = lds[i];
  }
  __syncthreads();
  // one elimination: the entry (i, j) after pivot k, from its old value, the
  // pivot row's and column's and the pivot's reciprocal (0: the variable leaves
  // the system)
  auto elim = [](int i, int j, int k, double pij, double pik, double pkj, double ip) {
    const double r = pkj * ip;
    return i == k ? (j == k ? ip : r) : j == k ? -pik * ip : pij - pik * r;
  };
  auto recip = [](double pv) { return pv > 1e-9 ? 1.0 / pv : 0.0; };
  const int gi = tid >> 6, gj = tid & 63;
  int cur = 0;
  for (int k = 0; k < nn; k += 2, cur ^= 1) {  // reads one copy, writes the other
    const double(*P)[MG_DENSE + 1] = A[cur];
    double(*Q)[MG_DENSE + 1] = A[cur ^ 1];
    if (gj < nn) {
      const int m = k + 1;
      const double ip = recip(P[k][k]), pkj = P[k][gj];
      if (m < nn) {
        const double pkm = P[k][m], pmk = P[m][k];
        const double im = recip(elim(m, m, k, P[m][m], pmk, pkm, ip));
        const double pmj = elim(m, gj, k, P[m][gj], pmk, pkj, ip);
        for (int i = gi; i < nn; i += ST / 64) {
          const double pik = P[i][k];
          const double v = elim(i, gj, k, P[i][gj], pik, pkj, ip);
          Q[i][gj] = elim(i, gj, m, v, elim(i, m, k, P[i][m], pik, pkm, ip), pmj, im);
        }
      } else {
        for (int i = gi; i < nn; i += ST / 64)
          Q[i][gj] = elim(i, gj, k, P[i][gj], P[i][k], pkj, ip);
      }
    }
    __syncthreads();
  }
  float *inv = pack + (d.tail < last ? (int)(l - lds) + 26 * nn : 0);
  for (int t = tid; t < nn * nn; t += ST) {
    const int i = t / nn, j = t % nn;
    global_mut(inv)[t] = (float)(A[cur][i][j] * sc[i] * sc[j]);
  }
}

// Over the coupled rows: the smallest row sum over diagonal, how many rows
// there are, how many whose row sum over diagonal exceeds `heavy`, and the sums of
// their row sums and diagonals (per block, then over the blocks to host memory):
// what the mass term leaves of the constant's energy.
constexpr int ROWSUMS = 5;
__global__ void __launch_bounds__(NT)
    mk_rowsum(int n, const int *__restrict__ row_bd, const int *__restrict__ sp,
              const double *__restrict__ sv, const double *__restrict__ diag, double heavy,
              double *__restrict__ out) {
  // the XCDs' rows are the solvers': entries that another XCD had read were slower
  // for all of the solve (P2 100^2: k_step 7.0 us instead of 5.9)
  const int i = xcd_block(blockIdx.x, gridDim.x) * NT + threadIdx.x;
  double v = 1.0, cnt[ROWSUMS - 1] = {};
  if (i < n && row_bd[i] < 0) {
    const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
    double sum = diag[i];
    bool coupled = false;
    for (int k = 0; k < w; k += 8) {
      double a[8];
#pragma unroll
      for (int u = 0; u < 8; u++)
        a[u] = __builtin_nontemporal_load(sv + off + 64 * min(k + u, w - 1));
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (k + u < w) {
          sum += a[u];
          coupled = coupled || a[u] != 0.0;
        }
    }
    v = sum / diag[i];
    cnt[0] = coupled;
    cnt[1] = coupled && v > heavy;
    cnt[2] = coupled ? sum : 0.0;
    cnt[3] = coupled ? diag[i] : 0.0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  __shared__ double sh[ROWSUMS][NT / 64];
  const int wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < ROWSUMS - 1; j++) cnt[j] = wave_sum(cnt[j]);
  if ((threadIdx.x & 63) == 0) {
    sh[0][wv] = v;
#pragma unroll
    for (int j = 0; j < ROWSUMS - 1; j++) sh[1 + j][wv] = cnt[j];
  }
  __syncthreads();
  if (threadIdx.x < ROWSUMS) {
    double t = sh[threadIdx.x][0];
    for (int k = 1; k < NT / 64; k++)
      t = threadIdx.x ? t + sh[threadIdx.x][k] : fmin(t, sh[0][k]);
    out[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
  }
}
__global__ void __launch_bounds__(RT)
    ms_rowsum(int G, const double *__restrict__ part, double *__restrict__ host) {
  double v = 1.0;
  for (int k = threadIdx.x; k < G; k += RT) v = fmin(v, part[k]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  __shared__ double sh[RT / 64];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  double cnt[ROWSUMS - 1];
  sum_partials<ROWSUMS - 1>(part + G, G, cnt);  // (its barrier covers sh)
  if (threadIdx.x == 0) {
    for (int k = 1; k < RT / 64; k++) v = fmin(v, sh[k]);
    host[0] = v;
#pragma unroll
    for (int j = 0; j < ROWSUMS - 1; j++) host[1 + j] = cnt[j];
  }
}

// ---------------------------------------------------------------- CG kernels

// A row's scaled residual for mk_lead, in FP64 and without the factor sc, which
// ms_start takes from all of them (in q, which mk_dir is the first to need).
__device__ __forceinline__ void leave_residual(const MgSys &d, int i, double ri) {
  global_mut(d.q)[i] = ri * global_ptr(d.dsq)[i];
}

// A row's residual after the first smoothing step, x0 - rs its negative
// without the off-diagonal part `dot`: with one step the input of the
// restriction, in the unscaled form's dual, sqrt(a_ii) (rs - Â x0), in the
// order of the cells; with two, the second step.
__device__ __forceinline__ void smooth_on(const MgSys &d, int i, float x0, float rs, double dot) {
  const double res = (double)rs - (double)x0 - dot;
  if (d.steps == 2) {
    global_mut(d.t)[i] = (float)((1.0 + (double)CM) * (double)x0 +
                                 (double)(C1 * global_ptr(d.minv)[i]) * res);
  } else {
    const int k = global_ptr(d.pos)[i];
    if (k >= 0) global_mut(d.ts)[k] = (float)(res * (double)global_ptr(d.sq)[i]);
  }
}

// Where the smoothing before the correction left its result.
__device__ __forceinline__ const float *smoothed(const MgSys &d) {
  return d.steps == 2 ? d.t : d.x0;
}

// Row i's product with the FP32 scaled off-diagonals.
template <class L, class F>
__device__ __forceinline__ double dot32(const MgSys &d, int i, L load, F comb) {
  return d.sd ? sell_dot16<float>(i, d.sp, d.sd, d.sv32, load, comb)
              : sell_dot<float>(i, d.sp, d.sc, d.sv32, load, comb);
}
template <class L>
__device__ __forceinline__ double dot32(const MgSys &d, int i, L load) {
  return dot32(d, i, load, [](float v) { return (double)v; });
}

// Start: x = b on identity rows and 0 elsewhere, r = b - A x (0 on those
// rows, b on the rest), p = 0; partials of r.r and b.b.  (b_ null: the
// descriptor's b.)
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
    const bool ident = i >= d.n || global_ptr(d.row_bd)[i] >= 0;
    const double ri = ident ? 0.0 : bi;
    global_mut(d.x)[i] = (ident && i < d.n) ? bi : 0.0;
    global_mut(d.p[0])[i] = 0.0;
    global_mut(d.p[1])[i] = 0.0;
    // never written for a row outside the grids, but read (times zero) through
    // its padding entries
    if (global_ptr(d.pos)[i] < 0) global_mut(d.t)[i] = 0.0f;
    global_mut(d.r[0])[i] = ri;
    leave_residual(d, i, ri);
    t[0] = ri * ri;
    t[1] = bi * bi;
  }
  put_partials<2>(t, d.part4, d.nblk, m.y);
}

__global__ void __launch_bounds__(RT)
    ms_start(const MgSys *__restrict__ D, MgScal *S_, const int *__restrict__ list, int sys,
             double rtol2, int maxit) {
  if (list) sys = list[blockIdx.x];
  const MgSys &d = D[sys];
  MgScal *S = S_ + sys;
  double t[2];
  sum_partials<2>(d.part4, d.nblk, t);
  if (threadIdx.x != 0) return;
  MgScal s{};
  s.bb = t[1];
  s.tol2 = rtol2 * t[1];
  s.maxit = maxit;
  s.true_prev = -1.0;
  // |sc r| in [1, 2) at the start; what is left of it at the end, 1e-16 of it at
  // the least, is far above FP32's smallest numbers
  const double s1 = *global_ptr(d.unit);
  s.sc = t[0] > 0.0 && isfinite(t[0]) ? ldexp(1.0, -ilogb(sqrt(t[0]))) : 1.0;
  s.back = s1 * s1 / s.sc;
  s.a.rr = t[0];
  s.a.first = 1;
  s.a.status = (!(t[0] == t[0]) || !isfinite(t[0])) ? ST_NAN
               : t[0] <= s.tol2                     ? ST_CONV
                                                    : ST_RUN;
  *S = s;
}

// The residual recomputed from the FP64 matrix once CG has stopped, in the
// form a restart continues from; partials of r.r.
__global__ void __launch_bounds__(NT)
    mk_check(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys,
             const double *b_) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status == ST_RUN || S[m.x].checked) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  double t[1] = {0.0};
  if (i < d.npad) {
    const gptr<double> x = global_ptr(d.x);
    const double bi = i < d.n ? global_ptr(b_ ? b_ : d.b)[i] : 0.0;
    const double ax = global_ptr(d.diag)[i] * x[i] +
                      sell_dot<double>(i, d.sp, d.sc, d.sv64, [&](int c) { return x[c]; });
    const double ri = bi - ax;
    global_mut(d.r[S[m.x].a.it & 1])[i] = ri;
    leave_residual(d, i, ri);
    t[0] = ri * ri;
  }
  put_partials<1>(t, d.part4, d.nblk, m.y);
}

// The recursive residual decides only when the true one agrees; otherwise CG
// restarts from the true one, eight times at most, and until |r|^2 falls by less
// than a tenth: then it is at the floor that rounding in x sets, eps |A| |x|, and
// the solve ends as converged, its residual in the stats, as FP64 Jacobi-PCG's
// does.  (Stopped at less than a factor of four, 23 of 468 solves with rtol 1 to
// 3 times their floor ended above rtol, by up to 11%; so do 4 now, by 2%, and 13
// of Jacobi-PCG's.)  host: a pinned copy of the state for the host (null: none).
__global__ void __launch_bounds__(RT)
    ms_check(const MgSys *__restrict__ D, MgScal *S_, const int *__restrict__ list, int sys,
             MgScal *host) {
  if (list) sys = list[blockIdx.x];
  if (sys < 0) return;
  MgScal *S = S_ + sys;
  if (S->a.status != ST_RUN && !S->checked) {  // (uniform: written at the end only)
    double t[1];
    sum_partials<1>(D[sys].part4, D[sys].nblk, t);
    if (threadIdx.x == 0) {
      const double rr = t[0];
      S->rr_true = rr;
      if (S->a.status == ST_CONV && !(rr <= S->tol2) && S->a.it < S->maxit && S->nrepl < 8 &&
          rr == rr && !(S->true_prev >= 0.0 && !(rr < 0.9 * S->true_prev))) {
        S->true_prev = rr;
        S->nrepl += 1;
        S->a.rr = rr;
        S->a.first = 1;
        S->a.status = ST_RUN;
      } else {
        if (S->a.status == ST_CONV && rr != rr) S->a.status = ST_NAN;
        S->checked = 1;
      }
    }
  }
  if (host && threadIdx.x == 0) host[sys] = *S;
}

// sum_small's input for systems with many partials: one block's sums.
template <int NV>
__global__ void __launch_bounds__(RT)
    ms_reduce(const MgSys *__restrict__ D, const MgScal *S, const int *__restrict__ list,
              int sys) {
  if (list) sys = list[blockIdx.x];
  if (sys < 0) return;
  const MgSys &d = D[sys];
  if (d.gsum == d.nblk || (NV == 1 ? S[sys].a : S[sys].b).status != ST_RUN) return;
  double t[NV];
  sum_partials<NV>(NV == 1 ? d.partz : d.part4, d.nblk, t);
  if (threadIdx.x == 0)
#pragma unroll
    for (int j = 0; j < NV; j++) global_mut(NV == 1 ? d.sumz : d.sum4)[j] = t[j];
}

// p = z + beta p (into the other buffer), q = A p, and r and q with the first
// smoothing step's weight for mk_step; partials of p.q, r.q, q.q, r.r.  A
// neighbour's p is formed on the fly by the same fused multiply-add as its own
// row forms it.
__global__ void __launch_bounds__(NT)
    mk_dir(const int2 *__restrict__ map, const MgSys *__restrict__ D, MgScal *S_, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0) return;
  const MgSys &d = D[m.x];
  MgScal *S = S_ + m.x;
  const bool lead = m.y == 0 && threadIdx.x == 0;
  MgState st = S->a;
  if (st.status != ST_RUN) {
    if (lead) S->b.status = st.status;
    return;
  }
  double rz[1];
  sum_small<1>(d.gsum == d.nblk ? d.partz : d.sumz, d.gsum, rz);
  const double back = S->back;  // z as the V-cycle left it -> z
  rz[0] *= back;
  st.status = rz[0] != rz[0] || !isfinite(rz[0]) ? ST_NAN : !(rz[0] > 0.0) ? ST_BREAK : ST_RUN;
  const double beta = st.first ? 0.0 : rz[0] / st.rz;
  st.rz = rz[0];
  if (lead) S->b = st;
  if (st.status != ST_RUN) return;
  const bool odd = st.it & 1;
  const gptr<double> p = global_ptr(d.p[odd]);
  const gptr<float> z = global_ptr(d.z);
  const int i = m.y * NT + threadIdx.x;
  double t[4] = {0.0, 0.0, 0.0, 0.0};
  if (i < d.npad) {
    struct zp { float z; double p; };
    auto load = [&](int c) { return zp{z[c], p[c]}; };
    auto comb = [&](zp v) { return fma(beta, v.p, (double)v.z * back); };
    const double pi = comb(load(i)), ri = global_ptr(d.r[odd])[i];
    const double qi =
        global_ptr(d.diag)[i] * pi + sell_dot<double>(i, d.sp, d.sc, d.sv64, load, comb);
    global_mut(d.p[!odd])[i] = pi;
    global_mut(d.q)[i] = qi;
    const double w = (double)((d.steps == 2 ? C0 : OM) * global_ptr(d.minv)[i]) *
                     global_ptr(d.dsq)[i] * S->sc;
    ((gmptr<f2_t>)reinterpret_cast<f2_t *>(d.wrq))[i] = f2_t{(float)(w * ri), (float)(w * qi)};
    t[0] = pi * qi;
    t[1] = ri * qi;
    t[2] = qi * qi;
    t[3] = ri * ri;
  }
  put_partials<4>(t, d.part4, d.nblk, m.y);
}

// x += alpha p, r -= alpha q (p: the buffer mk_dir wrote; r into the other
// buffer), and the next V-cycle's first smoothing step and residual.  The step
// of row and neighbours alike is w r - alpha w q from mk_dir's pair (w the
// step's weight), one 8-byte gather: against an update and a residual of their
// own it saves a launch, one pass of P1 64^2 1.11 -> 1.06 ms, heat 200^2 1.39 ->
// 1.35, even at 1024^2; with the neighbours' r, q and weights gathered (28
// bytes) 1024^2 was 1.3% slower.
__global__ void __launch_bounds__(NT)
    mk_step(const int2 *__restrict__ map, const MgSys *__restrict__ D, MgScal *S_, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0) return;
  const MgSys &d = D[m.x];
  MgScal *S = S_ + m.x;
  const bool lead = m.y == 0 && threadIdx.x == 0;
  MgState st = S->b;
  if (st.status != ST_RUN) {
    if (lead) S->a.status = st.status;
    return;
  }
  double t[4];
  sum_small<4>(d.gsum == d.nblk ? d.part4 : d.sum4, d.gsum, t);
  const double pq = t[0];
  const bool ok = pq > 0.0 && isfinite(pq);  // else NaN, or not SPD
  const double alpha = ok ? st.rz / pq : 0.0;
  st.it += 1;
  st.first = 0;
  st.rr = ok ? fmax(t[3] - 2.0 * alpha * t[1] + alpha * alpha * t[2], 0.0) : st.rr;
  st.status = pq != pq || isinf(pq) ? ST_NAN
              : !ok                 ? ST_BREAK
              : st.rr <= S->tol2    ? ST_CONV
              : st.it >= S->maxit   ? ST_MAXIT
                                    : ST_RUN;
  if (lead) S->a = st;
  const int i = m.y * NT + threadIdx.x;
  if (!ok || i >= d.npad) return;
  const double ri = fma(-alpha, global_ptr(d.q)[i], global_ptr(d.r[(st.it & 1) ^ 1])[i]);
  global_mut(d.x)[i] = fma(alpha, global_ptr(d.p[st.it & 1])[i], global_ptr(d.x)[i]);
  global_mut(d.r[st.it & 1])[i] = ri;
  if (st.status != ST_RUN) return;
  const gptr<f2_t> w = frac_ptr(d.wrq);
  auto load = [&](int c) { return w[c]; };
  auto first = [&](f2_t v) { return (float)fma(-alpha, (double)v.y, (double)v.x); };
  const float rs = (float)(ri * global_ptr(d.dsq)[i] * S->sc), x0 = first(load(i));
  global_mut(d.rs)[i] = rs;
  global_mut(d.x0)[i] = x0;
  smooth_on(d, i, x0, rs, dot32(d, i, load, [&](f2_t v) { return (double)first(v); }));
}

// The scaled residual, the first smoothing step and the residual after it from
// what mk_start or mk_check left, when CG starts.
__global__ void __launch_bounds__(NT)
    mk_lead(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN || !S[m.x].a.first) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  const gptr<double> q = global_ptr(d.q);
  const gptr<float> w = global_ptr(d.minv);
  const double sc = S[m.x].sc;
  const float om = d.steps == 2 ? C0 : OM;
  struct qw { double q; float w; };
  auto load = [&](int c) { return qw{q[c], w[c]}; };
  auto first = [&](qw v) { return om * v.w * (float)(v.q * sc); };
  const qw own = load(i);
  const float x0 = first(own), rs = (float)(own.q * sc);
  global_mut(d.rs)[i] = rs;
  global_mut(d.x0)[i] = x0;
  smooth_on(d, i, x0, rs, dot32(d, i, load, [&](qw v) { return (double)first(v); }));
}

// The first of two smoothing steps after the correction (steps = 2):
// x0 = t + C0 M^-1 (rs - Â t)
__global__ void __launch_bounds__(NT)
    mk_mid(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  const gptr<float> t = global_ptr(d.t);
  const double res = (double)global_ptr(d.rs)[i] - (double)t[i] -
                     dot32(d, i, [&](int c) { return t[c]; });
  global_mut(d.x0)[i] =
      (float)fma((double)(C0 * global_ptr(d.minv)[i]), res, (double)t[i]);
}

// ts = the fine residual after the second smoothing step (steps = 2)
__global__ void __launch_bounds__(NT)
    mk_res(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  if (i >= d.npad) return;
  const gptr<float> x = global_ptr(d.t);
  const double res = (double)global_ptr(d.rs)[i] - (double)x[i] -
                     dot32(d, i, [&](int c) { return x[c]; });
  const int k = global_ptr(d.pos)[i];
  if (k >= 0) global_mut(d.ts)[k] = (float)(res * (double)global_ptr(d.sq)[i]);
}

// One cell's share of node (X, Y) of the first grid in P^T t: the sum over
// the rows of cell (X - (q & 1), Y - (q >> 1)).
__device__ __forceinline__ double restrict_cell(const MgSys &d, const MgLevel &l, int X, int Y,
                                                int q) {
  const int ncx = l.nx - 1, ncy = l.ny - 1, cx = X - (q & 1), cy = Y - (q >> 1);
  if (cx < 0 || cx >= ncx || cy < 0 || cy >= ncy) return 0.0;
  const gptr<int> cptr = global_ptr(d.cptr);
  const gptr<f2_t> cfrac = frac_ptr(d.cfrac);
  const gptr<float> t = global_ptr(d.ts);
  const int c = cy * ncx + cx, k1 = cptr[c + 1];
  double s = 0.0;
  int k = cptr[c];
  for (; k + 3 < k1; k += 4) {  // four rows' loads in flight
    f2_t f[4];
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      f[u] = cfrac[k + u];
      v[u] = t[k + u];
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      s += (double)((q & 1 ? f[u].x : 1.0f - f[u].x) * (q >> 1 ? f[u].y : 1.0f - f[u].y)) *
           (double)v[u];
  }
  for (; k < k1; k++) {
    const f2_t f = cfrac[k];
    s += (double)((q & 1 ? f.x : 1.0f - f.x) * (q >> 1 ? f.y : 1.0f - f.y)) * (double)t[k];
  }
  return s;
}

// First grid: b = P^T t and the first smoothing step from zero; four threads
// a node, one for each of its cells.
__global__ void __launch_bounds__(NT)
    mk_restrict(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S,
                int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const MgLevel &l = d.lv[0];
  const int id = m.y * (NT / 4) + (threadIdx.x >> 2);
  const bool in = id < l.nx * l.ny;
  const int X = id % l.nx, Y = id / l.nx;
  double s = in ? restrict_cell(d, l, X, Y, threadIdx.x & 3) : 0.0;
  s += __shfl_xor(s, 1, 64);
  s += __shfl_xor(s, 2, 64);
  if (!in || (threadIdx.x & 3)) return;
  const int at = mg_at(l.px, X, Y);
  global_mut(l.b)[at] = (float)s;
  global_mut(l.x)[at] = OM * global_ptr(l.minv)[at] * (float)s;
}

// A grid node's product with its stencil; v: the node's value, pv its pitch.
template <class V>
__device__ __forceinline__ double stencil(const MgLevel &l, int at, V v, int pv) {
  const gptr<float> a = global_ptr(l.a);
  float c[25];
#pragma unroll
  for (int o = 0; o < 25; o++) c[o] = a[(size_t)o * l.pn + at];
  double s = 0.0;
#pragma unroll
  for (int o = 0; o < 25; o++)
    s += (double)c[o] * (double)v[(o / 5 - 2) * pv + o % 5 - 2];
  return s;
}

// Tiles of the grids above the tail: TC x TC nodes of the coarser grid, or
// TF x TF nodes of the finer one.  Both keep a block at one or two rounds of
// its threads, and the residuals (or corrected values) that neighbouring
// tiles both need are 13% of a tile's.
constexpr int TF = 16, TC = TF / 2, TT = 320;

// Grid k -> k + 1: residual b - A x of a tile (in LDS), restricted, with the
// coarser grid's first smoothing step from zero.
__global__ void __launch_bounds__(TT)
    gk_down(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys,
            int k) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN) return;
  const MgLevel &l = D[m.x].lv[k], &c = D[m.x].lv[k + 1];
  constexpr int W = TF + 1, WX = W + 2 * MG_HALO;  // residuals, values around
  __shared__ float xs[WX * WX], ts[W * W];
  const int ntx = (c.nx + TC - 1) / TC;
  const int X0 = m.y % ntx * TC, Y0 = m.y / ntx * TC;  // coarse corner
  const int x0 = 2 * X0 - 1, y0 = 2 * Y0 - 1;          // the residuals' corner
  for (int i = threadIdx.x; i < WX * WX; i += TT) {
    const int x = x0 - MG_HALO + i % WX, y = y0 - MG_HALO + i / WX;
    xs[i] = x >= 0 && x < l.nx && y >= 0 && y < l.ny ? global_ptr(l.x)[mg_at(l.px, x, y)] : 0.0f;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < W * W; i += TT) {
    const int ix = i % W, iy = i / W, x = x0 + ix, y = y0 + iy;
    float res = 0.0f;
    if (x >= 0 && x < l.nx && y >= 0 && y < l.ny) {
      const int at = mg_at(l.px, x, y);
      res = (float)((double)global_ptr(l.b)[at] -
                    stencil(l, at, xs + (iy + MG_HALO) * WX + ix + MG_HALO, WX));
    }
    ts[i] = res;
  }
  __syncthreads();
  if (threadIdx.x >= TC * TC) return;
  const int ix = threadIdx.x % TC, iy = threadIdx.x / TC, X = X0 + ix, Y = Y0 + iy;
  if (X >= c.nx || Y >= c.ny) return;
  const float *t = ts + (2 * iy + 1) * W + 2 * ix + 1;
  const float s = t[0] + 0.5f * ((t[-1] + t[1]) + (t[-W] + t[W])) +
                  0.25f * ((t[-W - 1] + t[-W + 1]) + (t[W - 1] + t[W + 1]));
  const int at = mg_at(c.px, X, Y);
  global_mut(c.b)[at] = s;
  global_mut(c.x)[at] = OM * global_ptr(c.minv)[at] * s;
}

// A grid's correction at node (x, y) of the finer grid.
template <class V>
__device__ __forceinline__ float prolong_at(V xc, int px, int x, int y) {
  const int at = mg_at(px, x >> 1, y >> 1), ax = x & 1, ay = y & 1;
  // the four nodes around (weights 1, 1/2 or 1/4)
  return 0.25f * ((xc[at] + xc[at + ax]) + (xc[at + ay * px] + xc[at + ay * px + ax]));
}

// Interpolation in a cell (v: its first node, pv the pitch).
template <class V>
__device__ __forceinline__ float bilinear(f2_t f, V v, int pv) {
  return (1.0f - f.x) * (1.0f - f.y) * v[0] + f.x * (1.0f - f.y) * v[1] +
         (1.0f - f.x) * f.y * v[pv] + f.x * f.y * v[pv + 1];
}

// Grid k: a tile's corrected values x + P t of grid k + 1 (in LDS), then
// t = those + w M^-1 (b - A those).  ROWS (k = 0): the smoothed values stay in LDS and
// the rows of the tile's cells take theirs, t = x0 + sqrt(a_ii) P x.
template <bool ROWS>
__global__ void __launch_bounds__(TT)
    gk_up(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys,
          int k) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const MgLevel &l = d.lv[k], &c = d.lv[k + 1];
  constexpr int W = ROWS ? TF + 1 : TF, WX = W + 2 * MG_HALO;
  __shared__ float ts[WX * WX], xs[ROWS ? W * W : 1];
  const int ntx = ((ROWS ? l.nx - 1 : l.nx) + TF - 1) / TF;
  const int x0 = m.y % ntx * TF, y0 = m.y / ntx * TF;
  for (int i = threadIdx.x; i < WX * WX; i += TT) {
    const int x = x0 - MG_HALO + i % WX, y = y0 - MG_HALO + i / WX;
    ts[i] = x >= 0 && x < l.nx && y >= 0 && y < l.ny
                ? global_ptr(l.x)[mg_at(l.px, x, y)] + prolong_at(global_ptr(c.t), c.px, x, y)
                : 0.0f;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < W * W; i += TT) {
    const int ix = i % W, iy = i / W, x = x0 + ix, y = y0 + iy;
    if (x >= l.nx || y >= l.ny) continue;
    const int at = mg_at(l.px, x, y);
    const float *t = ts + (iy + MG_HALO) * WX + ix + MG_HALO;
    const float res = (float)((double)global_ptr(l.b)[at] - stencil(l, at, t, WX));
    const float v = fmaf(OM * global_ptr(l.minv)[at], res, t[0]);
    // (x of this grid is still read by neighbouring tiles: t takes the result)
    if (ROWS) xs[i] = v;
    else global_mut(l.t)[at] = v;
  }
  if (!ROWS) return;
  __syncthreads();
  const int ncx = l.nx - 1, ncy = l.ny - 1;
  const gptr<int> cptr = global_ptr(d.cptr), crow = global_ptr(d.crow);
  const gptr<f2_t> cfrac = frac_ptr(d.cfrac);
  const gptr<float> x = global_ptr(smoothed(d));
  for (int i = threadIdx.x; i < TF * TF; i += TT) {
    const int ix = i % TF, iy = i / TF, cx = x0 + ix, cy = y0 + iy;
    if (cx >= ncx || cy >= ncy) continue;
    const int cl = cy * ncx + cx, k1 = cptr[cl + 1];
    for (int q = cptr[cl]; q < k1; q++) {
      const int r = crow[q];
      global_mut(d.t)[r] = fmaf(global_ptr(d.sq)[r], bilinear(cfrac[q], xs + iy * W + ix, W),
                                x[r]);
    }
  }
}

// A tail grid's product with its stencil, FP32 (at most MG_TAIL nodes: the
// cancellation costs three digits at most): v the node's value, pv its pitch.
template <class C>
__device__ __forceinline__ float stencil32(C c, const float *v, int pv) {
  float s = 0.0f;
#pragma unroll
  for (int o = 0; o < 25; o++) s = fmaf(c(o), v[(o / 5 - 2) * pv + o % 5 - 2], s);
  return s;
}

// The grids from d.tail on, in one workgroup.  A chain of some fifteen
// barriers, so latency is all: every stencil entry is requested before the
// first barrier, in quads (the first grid's into registers, TAIL_NODES nodes a
// thread; the others' into registers too, and on to LDS behind the first
// grid's residual), and the phases then run on LDS alone.  When every grid is
// in the tail it also restricts from the rows and interpolates to them.  LDS:
// x, b and t of every grid, entries and weights of all but the first, the
// dense inverse.  Of its 12.7 us at P2 101^2 (14.1 with the entries read one by
// one), 3.0 are the loads, 2.7 the first grid's two stencils, the rest phases of
// 0.25 - 0.7 us between barriers; P1 1024^2 13.7 -> 11.7 us.
constexpr int TAIL_NODES = MG_TAIL / RT;
constexpr int TAIL_PACK = 5;     // quads of the pack in flight, a thread
constexpr int TAIL_ROWS = 5;     // rows in flight, a thread
constexpr int TAIL_STAGE = 7000; // rows staged in LDS (12 bytes each), at most
constexpr int TAIL_LEVELS = 10;  // grids of a tail, at most
static_assert(TAIL_NODES * RT == MG_TAIL, "a thread owns whole nodes");
__global__ void __launch_bounds__(RT)
    mk_tail(const MgSys *__restrict__ D, const MgScal *S, const int *__restrict__ list, int sys) {
  if (list) sys = list[blockIdx.x];
  if (sys < 0 || S[sys].a.status != ST_RUN) return;
  extern __shared__ __align__(16) float lds[];
  __shared__ float part[RT / 64][64];
  const MgSys &d = D[sys];
  const int tid = threadIdx.x, first = d.tail, last = d.nlev - 1;
  const MgLevel &F = d.lv[first];
  const int fx = F.nx, nf = fx * F.ny;
  // the grids' sizes, kept in LDS: the descriptor's fields would be read from
  // memory in every phase
  struct Dim { int nx, ny, px, pn, nn; float inv; };
  __shared__ Dim dm[TAIL_LEVELS];
  if (tid <= last - first) {
    int nx = F.nx, ny = F.ny;
    for (int u = 0; u < tid; u++) {
      nx = mg_next(nx);
      ny = mg_next(ny);
    }
    dm[tid] = Dim{nx, ny, nx + 2 * MG_HALO, mg_pn(nx, ny), nx * ny, 1.0f / (float)nx};
  }
  __syncthreads();
  // (wave-uniform: scalar registers)
  auto dims = [&](int u) {
    const Dim q = dm[u];
    auto si = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    return Dim{si(q.nx), si(q.ny), si(q.px), si(q.pn), si(q.nn),
               __int_as_float(si(__float_as_int(q.inv)))};
  };
  const Dim d0 = dims(0);
  // node id -> position (exact: ids are far below 2^20)
  auto split = [](const Dim &q, int id, int &x, int &y) {
    y = (int)(((float)id + 0.5f) * q.inv);
    x = id - y * q.nx;
  };
  const int nu = last - first;  // the last grid's index in dm
  int tot = 0;
  for (int u = 0; u <= nu; u++) tot += dims(u).pn;
  float *coef = lds + 3 * tot;
  int npk = 0;  // the pack: entries and weights of the other grids, the inverse
  for (int u = 1; u <= nu; u++) npk += 26 * dims(u).nn;
  const float *cinv = coef + npk;
  npk = (npk + dims(nu).nn * dims(nu).nn + 3) & ~3;
  const gptr<f4_t> quad = (gptr<f4_t>)reinterpret_cast<const f4_t *>(d.pack);
  float ca[TAIL_NODES][28];
  int fat[TAIL_NODES];
#pragma unroll
  for (int u = 0; u < TAIL_NODES; u++) {
    const int id = min(tid + u * RT, nf - 1);
    int x, y;
    split(d0, id, x, y);
    fat[u] = mg_at(d0.px, x, y);
    if (__builtin_amdgcn_readfirstlane(tid) + u * RT >= nf) continue;  // none of the wave's
#pragma unroll
    for (int o = 0; o < 7; o++) {
      const f4_t v = quad[o * nf + id];
#pragma unroll
      for (int j = 0; j < 4; j++) ca[u][4 * o + j] = v[j];
    }
  }
  const gptr<f4_t> pk = quad + 7 * nf;
  f4_t pv[TAIL_PACK];
#pragma unroll
  for (int u = 0; u < TAIL_PACK; u++) pv[u] = pk[min(tid + u * RT, npk / 4 - 1)];
  for (int i = tid; i < 3 * tot / 4; i += RT)
    reinterpret_cast<f4_t *>(lds)[i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // (to LDS when the first grid's residual is done: nothing needs it before)
  auto put_pack = [&]() {
    f4_t *c4 = reinterpret_cast<f4_t *>(coef);
#pragma unroll
    for (int u = 0; u < TAIL_PACK; u++)
      if (tid + u * RT < npk / 4) c4[tid + u * RT] = pv[u];
    for (int i = tid + TAIL_PACK * RT; i < npk / 4; i += RT) c4[i] = pk[i];
  };
  // the first grid's right-hand side and first smoothing step from zero
  if (first == 0) {
    // each cell's rows (by way of LDS, where the pack goes later) into its
    // corners' shares; then the nodes' sums
    const int ncx = fx - 1, nc = ncx * (d0.ny - 1);
    const bool staged = d.n <= TAIL_STAGE;
    float *share = coef + (staged ? max(npk, 3 * d.n) : npk);  // [4][nc]
    float *row = coef;                        // [3][n]: value and position
    const gptr<f2_t> cfrac = frac_ptr(d.cfrac);
    const gptr<float> rt = global_ptr(d.ts);
    const gptr<int> cptr = global_ptr(d.cptr);
    const int n = d.n, nin = cptr[nc];  // rows that take part
    int k0[TAIL_NODES], k1[TAIL_NODES];
#pragma unroll
    for (int u = 0; u < TAIL_NODES; u++) {
      const int c = min(tid + u * RT, nc - 1);
      k0[u] = cptr[c];
      k1[u] = cptr[c + 1];
    }
    for (int i = staged ? tid : nin; i < nin; i += 4 * RT) {
      f2_t f[4];
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int j = min(i + u * RT, nin - 1);
        f[u] = cfrac[j];
        v[u] = rt[j];
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (i + u * RT < nin) {
          row[i + u * RT] = v[u];
          row[n + i + u * RT] = f[u].x;
          row[2 * n + i + u * RT] = f[u].y;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TAIL_NODES; u++) {
      const int c = tid + u * RT;
      if (c >= nc) continue;
      double s[4] = {0.0, 0.0, 0.0, 0.0};
      for (int k = k0[u]; k < k1[u]; k++) {
        float v, x, y;
        if (staged) {
          v = row[k];
          x = row[n + k];
          y = row[2 * n + k];
        } else {
          const f2_t f = cfrac[k];
          v = rt[k];
          x = f.x;
          y = f.y;
        }
        s[0] += (double)((1.0f - x) * (1.0f - y)) * (double)v;
        s[1] += (double)(x * (1.0f - y)) * (double)v;
        s[2] += (double)((1.0f - x) * y) * (double)v;
        s[3] += (double)(x * y) * (double)v;
      }
#pragma unroll
      for (int q = 0; q < 4; q++) share[q * nc + c] = (float)s[q];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TAIL_NODES; u++) {
      const int id = tid + u * RT;
      if (id >= nf) continue;
      int X, Y;
      split(d0, id, X, Y);
      float s = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int cx = X - (q & 1), cy = Y - (q >> 1);
        if (cx >= 0 && cx < ncx && cy >= 0 && cy < d0.ny - 1) s += share[q * nc + cy * ncx + cx];
      }
      lds[tot + fat[u]] = s;
      lds[fat[u]] = ca[u][25] * s;
    }
  } else {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TAIL_NODES; u++)
      if (tid + u * RT < nf) {
        lds[fat[u]] = global_ptr(F.x)[fat[u]];
        lds[tot + fat[u]] = global_ptr(F.b)[fat[u]];
      }
  }
  __syncthreads();
  int off = 0;
  const float *cf = coef;  // entries of the grid below the current one
  if (nu > 0) {
    float *x = lds, *b = x + tot, *t = b + tot;
#pragma unroll
    for (int v = 0; v < TAIL_NODES; v++)
      if (tid + v * RT < nf)
        t[fat[v]] = b[fat[v]] - stencil32([&](int o) { return ca[v][o]; }, x + fat[v], d0.px);
  }
  put_pack();
  __syncthreads();
  for (int u = 0; u < nu; u++) {  // down
    const Dim l = dims(u), c = dims(u + 1);
    float *x = lds + off, *b = x + tot, *t = b + tot;
    if (u > 0) {
      const float *cl = cf - 26 * l.nn;
      for (int id = tid; id < l.nn; id += RT) {
        int px, py;
        split(l, id, px, py);
        const int at = mg_at(l.px, px, py);
        t[at] = b[at] - stencil32([&](int o) { return cl[o * l.nn + id]; }, x + at, l.px);
      }
      __syncthreads();
    }
    float *xc = x + l.pn, *bc = xc + tot;
    for (int id = tid; id < c.nn; id += RT) {
      int X, Y;
      split(c, id, X, Y);
      const int at = mg_at(c.px, X, Y);
      const float *v = t + mg_at(l.px, 2 * X, 2 * Y);
      const float s = v[0] + 0.5f * ((v[-1] + v[1]) + (v[-l.px] + v[l.px])) +
                      0.25f * ((v[-l.px - 1] + v[-l.px + 1]) + (v[l.px - 1] + v[l.px + 1]));
      bc[at] = s;
      xc[at] = cf[25 * c.nn + id] * s;
    }
    __syncthreads();
    off += l.pn;
    cf += 26 * c.nn;
  }
  {  // last grid: the dense inverse (symmetric)
    const Dim q = dims(nu);
    const int lx = q.nx, nn = q.nn, px = q.px, i = tid & 63, g = tid >> 6;
    float *x = lds + off, *b = x + tot;
    float s = 0.0f;
    if (i < nn)
      for (int j = g; j < nn; j += RT / 64)
        s = fmaf(cinv[j * nn + i], b[mg_at(px, j % lx, j / lx)], s);
    part[g][i] = s;
    __syncthreads();
    if (tid < nn) {
      s = 0.0f;
#pragma unroll
      for (int g2 = 0; g2 < RT / 64; g2++) s += part[g2][tid];
      x[mg_at(px, tid % lx, tid / lx)] = s;
    }
    __syncthreads();
  }
  for (int u = nu - 1; u >= 0; u--) {  // up
    const Dim l = dims(u), c = dims(u + 1);
    off -= l.pn;
    cf -= 26 * c.nn;  // entries of grid u + 1; grid u's end there
    float *x = lds + off, *b = x + tot, *t = b + tot, *xc = x + l.pn;
    for (int id = tid; id < l.nn; id += RT) {
      int px, py;
      split(l, id, px, py);
      const int at = mg_at(l.px, px, py);
      t[at] = x[at] + prolong_at(xc, c.px, px, py);
    }
    __syncthreads();
    if (u == 0) break;
    const float *cl = cf - 26 * l.nn;
    for (int id = tid; id < l.nn; id += RT) {
      int px, py;
      split(l, id, px, py);
      const int at = mg_at(l.px, px, py);
      x[at] = fmaf(cl[25 * l.nn + id],
                   b[at] - stencil32([&](int o) { return cl[o * l.nn + id]; }, t + at, l.px),
                   t[at]);
    }
    __syncthreads();
  }
  const float *b0 = lds + tot, *t0 = b0 + tot;
  // the first grid's smoothing (a single grid has its solution already)
  auto smooth = [&](int v) {
    return nu > 0 ? fmaf(ca[v][25],
                         b0[fat[v]] -
                             stencil32([&](int o) { return ca[v][o]; }, t0 + fat[v], d0.px),
                         t0[fat[v]])
                  : lds[fat[v]];
  };
  if (first > 0) {
#pragma unroll
    for (int v = 0; v < TAIL_NODES; v++)
      if (tid + v * RT < nf) global_mut(F.t)[fat[v]] = smooth(v);
    return;
  }
  const gptr<int> cell = global_ptr(d.cell);
  const gptr<f2_t> frac = frac_ptr(d.frac);
  const gptr<float> sq = global_ptr(d.sq), x0 = global_ptr(smoothed(d));
  const float icx = 1.0f / (float)(fx - 1);
  int c[TAIL_ROWS];
  f2_t f[TAIL_ROWS];
  float w[TAIL_ROWS], y[TAIL_ROWS];
  auto rows = [&](int i) {  // TAIL_ROWS rows' loads in flight
#pragma unroll
    for (int u = 0; u < TAIL_ROWS; u++) {
      const int j = min(i + u * RT, d.npad - 1);
      c[u] = cell[j];
      f[u] = frac[j];
      w[u] = sq[j];
      y[u] = x0[j];
    }
  };
  rows(tid);
#pragma unroll
  for (int v = 0; v < TAIL_NODES; v++)
    if (nu > 0 && tid + v * RT < nf) lds[fat[v]] = smooth(v);
  __syncthreads();
  for (int i = tid; i < d.npad; i += TAIL_ROWS * RT) {
    if (i != tid) rows(i);
#pragma unroll
    for (int u = 0; u < TAIL_ROWS; u++) {
      if (i + u * RT >= d.npad || c[u] < 0) continue;
      const int cy = (int)(((float)c[u] + 0.5f) * icx);
      global_mut(d.t)[i + u * RT] =
          fmaf(w[u], bilinear(f[u], lds + mg_at(d0.px, c[u] - cy * (fx - 1), cy), d0.px), y[u]);
    }
  }
}

// z = S (t + w M^-1 (rs - Â t)), or the second step after mk_mid's; partials
// of r.z
__global__ void __launch_bounds__(NT)
    mk_post(const int2 *__restrict__ map, const MgSys *__restrict__ D, const MgScal *S, int sys) {
  const int2 m = where(map, sys);
  if (m.x < 0 || S[m.x].a.status != ST_RUN) return;
  const MgSys &d = D[m.x];
  const int i = m.y * NT + threadIdx.x;
  double v[1] = {0.0};
  if (i < d.npad) {
    float zi;
    if (d.steps == 2) {
      const gptr<float> x = global_ptr(d.x0);  // mk_mid's step
      const double xi = (double)x[i], res = (double)global_ptr(d.rs)[i] - xi -
                                            dot32(d, i, [&](int c) { return x[c]; });
      zi = (float)((xi + (double)CM * (xi - (double)global_ptr(d.t)[i]) +
                    (double)(C1 * global_ptr(d.minv)[i]) * res) * global_ptr(d.dsq)[i]);
    } else {
      const gptr<float> t = global_ptr(d.t);
      // a row outside the grids (Dirichlet, uncoupled) has no t: its value is x0
      const float ti = global_ptr(d.pos)[i] < 0 ? global_ptr(d.x0)[i] : t[i];
      const double res = (double)global_ptr(d.rs)[i] - (double)ti -
                         dot32(d, i, [&](int c) { return t[c]; });
      zi = (float)(fma((double)(OM * global_ptr(d.minv)[i]), res, (double)ti) *
                   global_ptr(d.dsq)[i]);
    }
    global_mut(d.z)[i] = zi;
    v[0] = global_ptr(d.r[S[m.x].a.it & 1])[i] * (double)zi;
  }
  put_partials<1>(v, d.partz, d.nblk, m.y);
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

// A mesh's dofs and how many others each shares an element with: P1 from the
// pattern (ptr, by internal node, with the diagonal), P2 from the number of
// incident elements (ptr, by the caller's dof): 3 for each of a vertex's, 3 and 2
// more for an edge's.  uid: row -> the caller's dof (null: the same).
struct DofGraph {
  const int *uid, *perm, *ptr;
  int degree, nnode;
  __device__ int neighbours(int i) const {
    const int u = uid ? uid[i] : i, v = degree == 1 ? perm[u] : u;
    const int k = ptr[v + 1] - ptr[v];
    return degree == 1 ? k - 1 : u < nnode ? 3 * k : 3 * k + 2;
  }
};

// Per block: the interior rows' bounding box, count, largest coupling extents
// (|dx|, |dy| over the matrix entries) and the sum over the rows of the part of
// their neighbours that the Dirichlet rows are.
__global__ void __launch_bounds__(NT)
    plan_extent(int n, const double2 *__restrict__ pt, const int *__restrict__ row_bd,
                const int *__restrict__ sp, const int *__restrict__ sc, DofGraph graph,
                double *__restrict__ out) {
  const int i = blockIdx.x * NT + threadIdx.x;
  // min x, min y, -max x, -max y, -max |dx|, -max |dy|
  double v[6] = {1e300, 1e300, 1e300, 1e300, 0.0, 0.0};
  double cnt[2] = {0.0, 0.0};
  if (i < n && takes_part(i, row_bd, sp, sc)) {
    const double2 a = pt[i];
    int coupled = 0;
    v[0] = a.x;
    v[1] = a.y;
    v[2] = -a.x;
    v[3] = -a.y;
    const int s0 = sp[i >> 6], w = (sp[(i >> 6) + 1] - s0) >> 6, off = s0 + (i & 63);
    for (int k = 0; k < w; k++) {
      const int j = sc[off + 64 * k];
      if (j >= n) continue;
      const double2 b = pt[j];
      v[4] = fmin(v[4], -fabs(a.x - b.x));
      v[5] = fmin(v[5], -fabs(a.y - b.y));
      coupled += j != i;
    }
    const int all = graph.neighbours(i);
    cnt[0] = 1.0;
    cnt[1] = all > coupled ? (double)(all - coupled) / all : 0.0;
  }
  __shared__ double sh[8][NT / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < 6; j++) {
    double t = v[j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t = fmin(t, __shfl_xor(t, o, 64));
    if (lane == 0) sh[j][wv] = t;
  }
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const double t = wave_sum(cnt[j]);
    if (lane == 0) sh[6 + j][wv] = t;
  }
  __syncthreads();
  if (threadIdx.x < 8) {
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
               const int *__restrict__ sp, const int *__restrict__ sc, double x0, double y0,
               double hx, double hy, int ncx, int ncy, int *__restrict__ cell,
               float2 *__restrict__ frac, int *__restrict__ key, int *__restrict__ row) {
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

// The rows' positions in the order of their cells.
__global__ void __launch_bounds__(NT)
    plan_cfrac(int n, int npad, const int *__restrict__ crow, const int *__restrict__ cell,
               const float2 *__restrict__ frac, float2 *__restrict__ cfrac,
               int *__restrict__ pos) {
  const int k = blockIdx.x * NT + threadIdx.x;
  if (k < n) {
    const int i = crow[k];
    cfrac[k] = frac[i];
    pos[i] = cell[i] < 0 ? -1 : k;
  } else if (k < npad) {
    pos[k] = -1;
  }
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
    pl->n = n;
    const unsigned g = nb(n, NT);
    DevBuf<double> ext((size_t)8 * g), ar(256);
    DevBuf<double2> pt(n);
    plan_points<<<g, NT, 0, st>>>(n, m.xy.p, own && s.degree == 2 ? s.d_dof_ends.p : nullptr,
                                  order, own ? nullptr : m.d_perm.p, m.nnode, m.d_edges.p,
                                  m.nedges, pt.p);
    const DofGraph graph{own ? s.d_uiperm() : order, m.d_perm.p,
                         m.degree == 1 ? m.d_rp.p : m.d_d2e_ptr.p, m.degree, m.nnode};
    plan_extent<<<g, NT, 0, st>>>(n, pt.p, s.d_row_bd.p, s.d_slice_ptr.p, s.d_sell_col.p, graph,
                                  ext.p);
    plan_area<<<256, NT, 0, st>>>(m.nelem, m.area.p, ar.p);
    HIPCHECK(hipGetLastError());
    std::vector<double> he((size_t)8 * g), ha(256);
    HIPCHECK(hipMemcpyAsync(he.data(), ext.p, ext.bytes(), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipMemcpyAsync(ha.data(), ar.p, ar.bytes(), hipMemcpyDeviceToHost, st));
    HIPCHECK(hipStreamSynchronize(st));
    double v[8] = {1e300, 1e300, 1e300, 1e300, 0, 0, 0, 0}, area = 0.0;
    for (int j = 0; j < 8; j++)
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
                                          s.d_sell_col.p, x0, y0, hx, hy, ncx, ncy,
                                          pl->cell.p, pl->frac.p, key.p, row.p);
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
    pl->cfrac.alloc(n);
    pl->pos.alloc(np);
    plan_cfrac<<<nb(np, NT), NT, 0, st>>>(n, np, pl->crow.p, pl->cell.p, pl->frac.p,
                                          pl->cfrac.p, pl->pos.p);
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
    // One fine smoothing step where the cells are wide against the couplings
    // (a uniform grid: 2; P1 forward + adjoint, one -> two steps: 150^2 1.44 ->
    // 1.61 ms, 300^2 1.78 -> 1.93, 700^2 even); else two (P1 jittered by a
    // fifth, 1.43: 100^2 1.55 -> 1.33 ms, 511^2 2.62 -> 2.42, 700^2 3.72 ->
    // 3.06; P2, 1: 101^2 3.47 -> 2.43 ms, 190^2 5.07 -> 3.44).
    pl->steps = hx > 1.6 * ex && hy > 1.6 * ey ? 1 : 2;
    int k = 0;
    pl->tail = -1;
    for (;; k++) {
      if (k == MG_MAXLEV) return pl;
      pl->nx[k] = nx;
      pl->ny[k] = ny;
      pl->px[k] = nx + 2 * MG_HALO;
      pl->pn[k] = mg_pn(nx, ny);
      if (pl->tail < 0 && pl->pn[k] <= MG_TAIL) pl->tail = k;
      if (nx * ny <= MG_DENSE) break;
      nx = mg_next(nx);
      ny = mg_next(ny);
    }
    pl->nlev = k + 1;
    if (pl->tail < 0 || pl->nlev - pl->tail > TAIL_LEVELS) return pl;
    // Where most rows neighbour a Dirichlet row Jacobi-PCG takes some 11 + 7 / F
    // iterations of 14 us (F: the part of their neighbours that are Dirichlet
    // rows), and the V-cycles' launches, two more for every grid above the tail,
    // cost more.  Forward + adjoint, Jacobi-PCG against multigrid CG: strips of
    // 2000 x 3 quads (F = 0.33, two grids) 1.00 and 1.12 ms, x 4 (0.22) 1.22 and
    // 1.14; 20000 x 3 (five grids) 1.07 and 1.80, x 6 (0.13) 1.98 and 2.10, x 8
    // (0.095) 2.57 and 2.18; every third row of 150^2 Dirichlet (one grid) 0.87 and
    // 1.08, every fourth 1.19 and 1.16.  P2, whose iterations are twice as many:
    // 5000 x 1 (0.75) 0.75 and 1.37, x 2 (0.35) 1.54 and 1.62, x 3 (0.21) 2.89 and
    // 2.09.  Without a grid above the tail multigrid CG is faster (200 x 2: 0.74 and
    // 0.63).
    const double near = std::max(0.125, 0.3 - 0.035 * pl->tail) * m.degree;
    if (pl->tail > 0 && v[7] > near * rows) return pl;
    pl->ok = true;
    return pl;
  } catch (...) {
    delete pl;
    throw;
  }
}

size_t tail_lds_of(const MgPlan &pl) {
  size_t t = 0, pack = 3;  // (whole quads)
  for (int k = pl.tail; k < pl.nlev; k++) {
    t += 3 * pl.pn[k];
    if (k > pl.tail) pack += (size_t)26 * pl.nx[k] * pl.ny[k];
  }
  const size_t nn = (size_t)pl.nx[pl.nlev - 1] * pl.ny[pl.nlev - 1];
  pack += nn * nn;
  if (pl.tail == 0)
    pack = std::max(pack, pl.n <= TAIL_STAGE ? (size_t)3 * pl.n : 0) +
           4 * (size_t)(pl.nx[0] - 1) * (pl.ny[0] - 1);
  return (t + pack) * sizeof(float);
}

}  // namespace

size_t mg_tail_lds(const MgPlan &pl) { return tail_lds_of(pl); }

size_t mg_setup_lds(const MgPlan &pl) {
  size_t t = pl.tail + 1 == pl.nlev ? (size_t)25 * pl.nx[pl.tail] * pl.ny[pl.tail] : 0;
  for (int k = pl.tail + 1; k < pl.nlev; k++) t += (size_t)26 * pl.nx[k] * pl.ny[k];
  return t * sizeof(float);
}

void mg_allow_lds(const MgPlan &pl) {
  const size_t lds = mg_tail_lds(pl);
  REQUIRE(lds <= 150 * 1024, ADMFEM_ERR_UNSUPPORTED, "tail grids too large for LDS");
  REQUIRE(mg_setup_lds(pl) <= 110 * 1024, ADMFEM_ERR_UNSUPPORTED, "tail grids too large for LDS");
  HIPCHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(mk_tail),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));
  HIPCHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(mk_tail_setup),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 110 * 1024));
}

void mg_plan_free(MgPlan *p) { delete p; }

static std::mutex g_plan;  // an engine and a solver may share the system

const MgPlan *mg_plan(System &s, hipStream_t st) {
  std::lock_guard<std::mutex> g(g_plan);
  if (!s.mg_plan && s.mesh) s.mg_plan = build_plan(s, *s.mesh, nullptr, st);
  else if (!s.mg_plan && s.mg_mesh) s.mg_plan = build_plan(s, *s.mg_mesh, s.mg_order, st);
  return s.mg_plan && s.mg_plan->ok ? s.mg_plan : nullptr;
}

// (false: a plan was made and does not suit the rows)
static bool mg_may_suit(const System &s) {
  std::lock_guard<std::mutex> g(g_plan);
  return !s.mg_plan || s.mg_plan->ok;
}

size_t mg_grid_floats(const MgPlan &pl) {
  size_t f = 0;
  for (int k = 0; k < pl.nlev; k++)
    f += (size_t)29 * pl.pn[k] +
         (k > pl.tail ? (size_t)26 * pl.nx[k] * pl.ny[k]
                      : k == pl.tail ? (size_t)28 * pl.nx[k] * pl.ny[k] : 0);
  return f + MG_DENSE * MG_DENSE + 3;
}

void mg_grid_layout(const MgPlan &pl, float *base, MgSys &d) {
  d.cell = pl.cell.p;
  d.frac = pl.frac.p;
  d.cptr = pl.cptr.p;
  d.crow = pl.crow.p;
  d.cfrac = pl.cfrac.p;
  d.pos = pl.pos.p;
  d.steps = pl.steps;
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
  d.pack = base;
}

void mg_parts(MgSys &d, int nblk, bool reduce, double *part) {
  d.nblk = nblk;
  d.part4 = part;
  d.partz = part + 4 * (size_t)nblk;
  d.sum4 = d.partz + nblk;
  d.sumz = d.sum4 + 4;
  d.unit = d.sumz + 1;
  d.gsum = reduce ? 1 : nblk;
}

struct MgWork {
  MgSys h{};                     // the descriptor (host copy)
  DevBuf<MgSys> d;
  DevBuf<MgScal> sc;
  MgScal *h_sc = nullptr;        // pinned
  DevBuf<double> x, r, r1, q, p0, p1, dsq, part;
  DevBuf<float2> wrq;
  DevBuf<float> sv32, sq, minv, z, rs, x0, t, ts, grid;
  int nblk = 0;
  int last_it = 14;              // iterations of the last solve
  uint64_t version = 0;          // of the matrix the set-up was made from
  ~MgWork() {
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
    w->r1.alloc(np);
    w->q.alloc(np);
    w->p0.alloc(np);
    w->p1.alloc(np);
    w->dsq.alloc(np);
    w->part.alloc((size_t)5 * w->nblk + 6);
    w->sv32.alloc(std::max(1, s.slice_ptr.back()));
    w->sq.alloc(np);
    w->minv.alloc(np);
    w->z.alloc(np);
    w->rs.alloc(np);
    w->x0.alloc(np);
    w->t.alloc(np);
    w->ts.alloc(np);
    w->wrq.alloc(np);
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
    d.r[0] = w->r.p;
    d.r[1] = w->r1.p;
    d.q = w->q.p;
    d.p[0] = w->p0.p;
    d.p[1] = w->p1.p;
    d.z = w->z.p;
    d.rs = w->rs.p;
    d.x0 = w->x0.p;
    d.t = w->t.p;
    d.ts = w->ts.p;
    d.wrq = w->wrq.p;
    d.n = s.n;
    d.npad = s.npad;
    mg_parts(d, w->nblk, w->nblk > MG_SUM, w->part.p);
    mg_grid_layout(pl, w->grid.p, d);
    mg_allow_lds(pl);
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

// ----------------------------------------------------------------- batches

static int mg_tiles_down(const MgPlan &pl, int k) {
  return (int)(nb(pl.nx[k + 1], TC) * nb(pl.ny[k + 1], TC));
}
static int mg_blocks_setup(const MgPlan &pl, int k) {
  const int64_t nf = (int64_t)pl.nx[k] * pl.ny[k];
  return (int)nb(k + 1 < pl.nlev ? std::max(nf, 4 * (int64_t)pl.nx[k + 1] * pl.ny[k + 1]) : nf, GS);
}
static int mg_tiles_up(const MgPlan &pl, int k) {
  return k ? (int)(nb(pl.nx[k], TF) * nb(pl.ny[k], TF))
           : (int)(nb(pl.nx[k] - 1, TF) * nb(pl.ny[k] - 1, TF));
}

void mg_stages(const MgPlan &pl, int npad, int (&nblk)[MG_STAGES]) {
  for (int &v : nblk) v = 0;
  nblk[MGS_ROWS] = (int)nb(npad, NT);
  if (pl.steps == 2) nblk[MGS_TWO] = nblk[MGS_ROWS];
  nblk[MGS_GALERKIN] = (int)nb((int64_t)pl.nx[0] * pl.ny[0], mg_gn(1));
  if (pl.tail > 0) nblk[MGS_RESTRICT] = (int)nb((int64_t)pl.nx[0] * pl.ny[0], NT / 4);
  for (int k = 0; k <= pl.tail; k++) nblk[MGS_SETUP + k] = mg_blocks_setup(pl, k);
  for (int k = 0; k < pl.tail; k++) {
    nblk[MGS_DOWN + k] = mg_tiles_down(pl, k);
    nblk[MGS_UP + k] = mg_tiles_up(pl, k);
  }
}

void mg_batch_setup(const MgBatch &B, const MgSys *D, hipStream_t st) {
  auto n = [&](int q) { return (unsigned)B.nmap[q]; };
  mk_scale<<<n(MGS_ROWS), NT, 0, st>>>(B.map[MGS_ROWS], D, 0);
  mk_galerkin<1><<<n(MGS_GALERKIN), GT, 0, st>>>(B.map[MGS_GALERKIN], D, 0);
  for (int k = 0; k <= B.tail; k++)
    gk_setup<<<n(MGS_SETUP + k), GS, 0, st>>>(B.map[MGS_SETUP + k], D, 0, k);
  mk_tail_setup<<<(unsigned)B.nsys, ST, B.setup_lds, st>>>(D, B.list, 0);
  HIPCHECK(hipGetLastError());
}

void mg_batch_start(const MgBatch &B, const MgSys *D, MgScal *S, double rtol2, int maxit,
                    hipStream_t st) {
  mk_start<<<(unsigned)B.nmap[MGS_ROWS], NT, 0, st>>>(B.map[MGS_ROWS], D, 0, nullptr);
  ms_start<<<(unsigned)B.nsys, RT, 0, st>>>(D, S, B.list, 0, rtol2, maxit);
  HIPCHECK(hipGetLastError());
}

void mg_batch_iterations(const MgBatch &B, const MgSys *D, MgScal *S, int iters, MgScal *host,
                         hipStream_t st) {
  auto n = [&](int q) { return (unsigned)B.nmap[q]; };
  const int2 *rows = B.map[MGS_ROWS];
  const unsigned nl = (unsigned)B.nsys, nr = n(MGS_ROWS);
  mk_lead<<<nr, NT, 0, st>>>(rows, D, S, 0);
  for (int it = 0; it < iters; it++) {
    if (n(MGS_TWO)) mk_res<<<n(MGS_TWO), NT, 0, st>>>(B.map[MGS_TWO], D, S, 0);
    if (B.tail > 0)
      mk_restrict<<<n(MGS_RESTRICT), NT, 0, st>>>(B.map[MGS_RESTRICT], D, S, 0);
    for (int k = 0; k < B.tail; k++)
      gk_down<<<n(MGS_DOWN + k), TT, 0, st>>>(B.map[MGS_DOWN + k], D, S, 0, k);
    mk_tail<<<nl, RT, B.tail_lds, st>>>(D, S, B.list, 0);
    for (int k = B.tail - 1; k > 0; k--)
      gk_up<false><<<n(MGS_UP + k), TT, 0, st>>>(B.map[MGS_UP + k], D, S, 0, k);
    if (B.tail > 0) gk_up<true><<<n(MGS_UP), TT, 0, st>>>(B.map[MGS_UP], D, S, 0, 0);
    if (n(MGS_TWO)) mk_mid<<<n(MGS_TWO), NT, 0, st>>>(B.map[MGS_TWO], D, S, 0);
    mk_post<<<nr, NT, 0, st>>>(rows, D, S, 0);
    if (B.reduce) ms_reduce<1><<<nl, RT, 0, st>>>(D, S, B.list, 0);
    mk_dir<<<nr, NT, 0, st>>>(rows, D, S, 0);
    if (B.reduce) ms_reduce<4><<<nl, RT, 0, st>>>(D, S, B.list, 0);
    mk_step<<<nr, NT, 0, st>>>(rows, D, S, 0);
  }
  mk_check<<<nr, NT, 0, st>>>(rows, D, S, 0, nullptr);
  ms_check<<<nl, RT, 0, st>>>(D, S, B.list, 0, host);
  HIPCHECK(hipGetLastError());
}

// The set-up of one matrix (descriptor `sys` of D): fine scaling, the grids'
// matrices and smoothing weights, the last grid's inverse.
void mg_setup(const MgPlan &pl, int nblk, const MgSys *D, int sys, hipStream_t st) {
  mk_scale<<<nblk, NT, 0, st>>>(nullptr, D, sys);
  const int64_t nodes = (int64_t)pl.nx[0] * pl.ny[0];
  if (nodes <= GALERKIN_SPLIT) mk_galerkin<4><<<nb(nodes, mg_gn(4)), GT, 0, st>>>(nullptr, D, sys);
  else mk_galerkin<1><<<nb(nodes, mg_gn(1)), GT, 0, st>>>(nullptr, D, sys);
  for (int k = 0; k <= pl.tail; k++)
    gk_setup<<<mg_blocks_setup(pl, k), GS, 0, st>>>(nullptr, D, sys, k);
  mk_tail_setup<<<1, ST, mg_setup_lds(pl), st>>>(D, nullptr, sys);
  HIPCHECK(hipGetLastError());
}

namespace {

void iteration(const MgPlan &pl, MgWork *w, hipStream_t st) {
  const MgSys *D = w->d.p;
  MgScal *S = w->sc.p;
  if (pl.steps == 2) mk_res<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  if (pl.tail > 0)
    mk_restrict<<<nb(pl.nx[0] * pl.ny[0], NT / 4), NT, 0, st>>>(nullptr, D, S, 0);
  for (int k = 0; k < pl.tail; k++)
    gk_down<<<mg_tiles_down(pl, k), TT, 0, st>>>(nullptr, D, S, 0, k);
  mk_tail<<<1, RT, mg_tail_lds(pl), st>>>(D, S, nullptr, 0);
  for (int k = pl.tail - 1; k > 0; k--)
    gk_up<false><<<mg_tiles_up(pl, k), TT, 0, st>>>(nullptr, D, S, 0, k);
  if (pl.tail > 0) gk_up<true><<<mg_tiles_up(pl, 0), TT, 0, st>>>(nullptr, D, S, 0, 0);
  if (pl.steps == 2) mk_mid<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  mk_post<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  if (w->nblk > MG_SUM) ms_reduce<1><<<1, RT, 0, st>>>(D, S, nullptr, 0);
  mk_dir<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
  if (w->nblk > MG_SUM) ms_reduce<4><<<1, RT, 0, st>>>(D, S, nullptr, 0);
  mk_step<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
}

// Whether the V-cycle suits the assembled matrix: not when a mass term
// dominates it.  Jacobi-PCG's condition number is about 2 over the smallest
// row sum over diagonal (1 for a lumped mass matrix, O(h^2) for a stiffness
// matrix); at 0.2 it needs about as many launches as the V-cycles do, and at three
// quarters of that for each grid above the tail, whose launches come on top (of
// about the number below): forward + adjoint of P1 heat steps, Jacobi-PCG against
// multigrid CG, 40^2 dt 1e-4 0.84 and 0.73 ms, 128^2 1e-5 1.04 and 1.05, 3e-5 1.43
// and 1.03, 400^2 1e-6 1.34 and 1.45, 3e-6 2.02 and 1.45.  P2's row sums say
// nothing one by one (a vertex function's integral is 0); over all rows their sum
// is 1.6 times the diagonals' for a mass matrix, and at half of that the two are
// even: 100^2 dt 1e-6 1.02 and 1.28, 3e-6 1.48 and 1.46; 40^2 (6,561 rows) 3e-6 0.95
// and 1.05, 3e-5 1.42 and 1.17; with few rows multigrid CG is the faster (20^2,
// 1,681, at any step: 0.96 and 0.90).
// A caller's matrix stays with Jacobi-PCG also where half its coupled rows
// have a row sum over diagonal above MASS_HEAVY / rows: mass outweighs
// stiffness even at the scale of the whole domain (0.25 / (dt kappa) for a heat
// step on P1, 0.19 on P2: dt below 4e-3 or 3e-3).  Gradients of such a step are
// differences of nearly equal fields, and their error at a given rtol depends on
// the solver.  Gradient in kappa against 64 bits, operator chain at rtol 1e-12 with
// boundary values of order 1, Jacobi-PCG and multigrid CG: dt 1e-4 P1 128^2 4.6e-9
// and 6.0e-9, 160^2 7.4e-9 and 8.1e-9 (64^2 1.1e-9 and 6.9e-10, P2 40^2 2.2e-9 and
// 7.2e-10), 3e-4 128^2 2.4e-9 and 4.7e-10, 1e-3 1.3e-9 and 4.1e-10, 3e-3 4.5e-10 and
// 3.1e-10.  So the line keeps the shortest steps as near as they were, and is wider
// than that takes: from 3e-4 on multigrid CG is the nearer and the faster (128^2 at
// 1e-3: 8.3 and 3.0 ms a chain, 160^2 9.2 and 3.0, P2 40^2 8.2 and 3.3).  Systems of
// the fused path and the engine, whose boundary rows are solved exactly, have no such
// line.
constexpr double MASS_DOMINANT = 0.2, MASS_DOMINANT_P2 = 0.8, MASS_HEAVY = 60.0;
constexpr int MASS_P2_ROWS = 4000;
// (Looked at before the plan, which a matrix that stays with Jacobi-PCG never
// needs: 0.3 ms on every new mesh.)
bool mg_pays(System &s, hipStream_t st) {
  if (!s.mass) return true;
  if (s.mg_pays_version != s.a_version) {
    const unsigned g = (nb(s.n, NT) + 7) / 8 * 8;
    if (!s.mg_rows.p) s.mg_rows.alloc(ROWSUMS * (size_t)g);
    mk_rowsum<<<g, NT, 0, st>>>(s.n, s.d_row_bd.p, s.d_slice_ptr.p, s.d_sell_val.p, s.d_diag.p,
                                MASS_HEAVY / s.n, s.mg_rows.p);
    HostSlot h(st);
    ms_rowsum<<<1, RT, 0, st>>>((int)g, s.mg_rows.p, h.written());
    HIPCHECK(hipGetLastError());
    h.wait();
    const bool callers = s.mesh == nullptr;
    const int degree = (callers ? s.mg_mesh : s.mesh)->degree;
    double least = MASS_DOMINANT;
    for (double nodes = s.n / 4.0; nodes > MG_TAIL - 350; nodes /= 4) least *= 0.75;
    const double rows = h.get<double>(8), heavy = h.get<double>(16), sum = h.get<double>(24),
                 diag = h.get<double>(32);
    s.mg_pays = !(h.get<double>(0) > least) && !(callers && 2.0 * heavy > rows) &&
                !(degree == 2 && s.n > MASS_P2_ROWS && sum > MASS_DOMINANT_P2 * diag);
    s.mg_pays_version = s.a_version;
  }
  return s.mg_pays;
}

}  // namespace

// Device memory of a plan and its work, about, per row (P1).
constexpr int MG_ROW_BYTES = 188;

// A sparse system's rows are the dofs of mesh m (m null: unknown, and it is
// Jacobi-PCG's), row i the caller's order[i]; both are only looked at in the
// solve that follows.  Its plan is kept for as long as the mesh stays the same
// one.
void mg_set_mesh(System &s, const Mesh *m, const int *order) {
  s.mg_off = !m || m->ndof != s.n || s.n < MG_MIN_ROWS;
  if (s.mg_off) return;
  s.mass = true;  // the matrix is the caller's: look before using the grids
  s.mg_mesh = m;
  s.mg_order = order;
  if (s.mg_serial == m->serial) return;
  if (s.mg_work) mg_work_free(s.mg_work);
  if (s.mg_plan) mg_plan_free(s.mg_plan);
  s.mg_work = nullptr;
  s.mg_plan = nullptr;
  s.mg_serial = m->serial;
}

// Solves by multigrid CG when that suits the system; false when it is
// Jacobi-PCG's: also when multigrid CG broke down, met a NaN or ran out of
// iterations or memory (MG_ROW_BYTES against 120), which Jacobi-PCG need not (and
// if it does, the status is its own).
bool mg_solve(System &s, const double *b, double *x_out, const admfem_solve_opts &o,
              admfem_solve_stats &stats, hipStream_t st) {
  if (s.mg_off || s.n < MG_MIN_ROWS || s.mg_failed == s.a_version) return false;
  auto t0 = std::chrono::steady_clock::now();
  if (!mg_may_suit(s)) return false;
  if (!mg_pays(s, st)) return false;
  // (memory is looked at where it is no small matter)
  const size_t need = (size_t)MG_ROW_BYTES * s.npad;
  if (!s.mg_work && need > (size_t)32 << 20 && need > device_available()) return false;
  const MgPlan *plan = nullptr;
  MgWork *w = nullptr;
  try {
    plan = mg_plan(s, st);
    if (!plan) return false;
    w = ensure_work(s, *plan, st);
  } catch (const OutOfMemory &) {
    release_device_memory();  // (others may need it as well)
    return false;
  }
  const MgPlan &pl = *plan;
  const MgSys *D = w->d.p;
  MgScal *S = w->sc.p;
  if (w->version != s.a_version) {  // a new matrix
    mg_setup(pl, w->nblk, D, 0, st);
    w->version = s.a_version;
  }
  mk_start<<<w->nblk, NT, 0, st>>>(nullptr, D, 0, b);
  ms_start<<<1, RT, 0, st>>>(D, S, nullptr, 0, o.rtol * o.rtol,
                             std::min(MG_GIVE_UP, std::max(1, o.max_iter / MG_PRODUCTS)));
  // Iterations are enqueued in chunks, each followed by the check (a no-op
  // while CG runs), and the host reads the state between chunks; kernels past
  // the end return at once.  The first chunk is what the system's last solve
  // took: the adjoint usually takes what the forward did.  Plain launches: the
  // host queues them faster than the device starts them, replayed graphs
  // measured the same (64^2 1.09 against 1.10 ms, 1024^2 5.02 against 5.06),
  // and a capture costs a first solve 0.2 - 3 ms and stops other threads' copies.
  // A longer interval than that only adds launches that do nothing (check_every
  // 1000 at 64^2: 21 ms instead of 0.4).
  const int most = o.check_every > 0 ? o.check_every : INT_MAX;
  int chunk = std::min(most, w->last_it);
  for (;;) {
    mk_lead<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0);
    for (int it = 0; it < chunk; it++) iteration(pl, w, st);
    mk_check<<<w->nblk, NT, 0, st>>>(nullptr, D, S, 0, b);
    ms_check<<<1, RT, 0, st>>>(D, S, nullptr, 0, w->h_sc);
    HIPCHECK(hipGetLastError());
    // (the solution as far as it is: no second wait for the final one, unless
    // it goes where the right-hand side still is)
    if (x_out != b)
      HIPCHECK(hipMemcpyAsync(x_out, w->x.p, sizeof(double) * s.n, hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipStreamSynchronize(st));
    if (w->h_sc->a.status != ST_RUN) break;
    chunk = std::min(most, 2);
  }
  if (w->h_sc->a.status != ST_CONV) {
    s.mg_failed = s.a_version;
    return false;
  }
  w->last_it = std::min(64, std::max(4, w->h_sc->a.it));
  if (x_out == b) {
    HIPCHECK(hipMemcpyAsync(x_out, w->x.p, sizeof(double) * s.n, hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipStreamSynchronize(st));
  }
  const MgScal &h = *w->h_sc;
  stats.iterations = MG_PRODUCTS * h.a.it;
  stats.replacements = h.nrepl;
  stats.rel_residual = h.bb > 0 ? std::sqrt(h.rr_true / h.bb) : 0.0;
  stats.status = ADMFEM_OK;
  stats.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return true;
}

}  // namespace admfem
