// Multigrid-preconditioned CG for mesh systems (mg.hip): structures shared by
// the single-system solver and the serving engine.
#pragma once
#include "internal.h"

namespace admfem {

constexpr int MG_MAXLEV = 16;    // grid levels at most
constexpr int MG_HALO = 2;       // nodes around a grid (the stencils reach 2)
constexpr int MG_TAIL = 2048;    // padded nodes of the first level of the tail kernel
constexpr int MG_DENSE = 49;     // nodes of the last level at most (dense inverse)

// One grid level: nx x ny nodes stored with room for MG_HALO nodes on every side
// (pitch px, pn entries in all), node (x, y) at mg_at.  In memory that room is
// neither written nor read; it is zero in the tail kernel's copies in LDS.
struct MgLevel {
  float *a;     // 25 planes of pn: the stencil entries, offset (dx, dy) at
                // plane (dy + 2) * 5 + dx + 2
  float *minv;  // smoother's weights
  float *x, *b, *t;
  int nx, ny, px, pn;
};
__host__ __device__ inline int mg_at(int px, int x, int y) {
  return (y + MG_HALO) * px + x + MG_HALO;
}

// Systems below this many rows stay with Jacobi-PCG.  One Poisson forward +
// adjoint, FP64, Jacobi-PCG -> multigrid CG: 50^2 5.6 -> 1.1 ms, 32^2 4.7 -> 1.0
// ms, 20^2 2.6 -> 0.93 ms, 14^2 1.6 -> 0.83 ms; at 12^2 and below the two are
// even.
constexpr int MG_MIN_ROWS = 200;

// Products with the system's matrix in an iteration (mk_step, mk_post,
// mk_dir): what max_iter bounds and the stats report, as for Jacobi-PCG, whose
// iterations are one product each.
constexpr int MG_PRODUCTS = 3;

// Iterations after which a solve is Jacobi-PCG's after all.  Coefficients or
// elements that the grids know nothing of slow both down, Jacobi-PCG more (P1
// 64^2 with white noise of deviation 5 in log kappa: 406 against 5,243; elements
// of 100 : 1: 110 against 740), so the line only ends what does not converge.
constexpr int MG_GIVE_UP = 2000;

// a grid's nodes along a side on the next one; its padded size
__host__ __device__ inline int mg_next(int n) { return n / 2 + 1; }
__host__ __device__ inline int mg_pn(int nx, int ny) {
  return ((nx + 2 * MG_HALO) * (ny + 2 * MG_HALO) + 63) / 64 * 64;
}

// One system: its matrix, the plan's arrays (shared by every system of the
// topology) and its vectors (internal row order, npad long).
struct MgSys {
  const int *sp, *sc;       // SELL slice offsets / columns
  const int16_t *sd;        // the columns as 16-bit offsets from the row, or null
  const int *row_bd;
  const double *sv64, *diag;  // FP64 matrix
  float *sv32;              // scaled off-diagonals a_ij / sqrt(a_ii a_jj)
  double *unit;             // s: the V-cycle works on s^2 A, a power of two
  double *dsq;              // 1 / (s sqrt(a_ii))
  float *sq, *minv;         // s sqrt(a_ii), smoother's weights
  const int *cell;          // grid cell of each row (-1: not interpolated)
  const float2 *frac;       // position inside the cell
  const int *cptr, *crow;   // rows by cell
  const float2 *cfrac;      // frac in that order
  const int *pos;           // each row's place in it (-1: none)
  const double *b;          // right-hand side
  double *x, *r[2], *q, *p[2];  // (r, p: iteration it reads one and writes the
                            // other; r[it & 1] is the residual after it)
  float *z, *rs, *x0, *t;   // preconditioned residual, scaled residual,
                            // smoothed correction, corrected
  float2 *wrq;              // r and q times the first smoothing step's weight
  float *ts;                // the restriction's input, in the cells' order
  double *part4, *partz;    // 4 x nblk and nblk block partials
  double *sum4, *sumz;      // their sums, when one block makes them
  int gsum;                 // values the wide kernels sum: nblk, or 1
  // the tail's matrices: its first grid's entries and weights as 7 quads a
  // node ([7][nodes], entry 25 the weight), then each further grid's [25][nodes]
  // and [nodes], then the dense inverse of the last
  float *pack;
  int n, npad, nblk;
  int nlev, tail;           // grid levels, first one of the tail kernel
  int steps;                // fine smoothing steps before and after (1 or 2)
  MgLevel lv[MG_MAXLEV];
};

// One system's solve: the state, in two copies (mk_dir reads a and writes b,
// mk_step reads b and writes a, every other kernel reads a).
struct MgState {
  double rz, rr;
  int status;               // as in cg.hip: 0 run, 1 converged, 2 iterations
                            // spent, 3 NaN, 4 breakdown
  int it, first;
};
struct MgScal {
  double bb, tol2;
  double rr_true, true_prev;  // |b - A x|^2 when CG last stopped, and before
  double sc, back;          // the V-cycle takes sc r and leaves z / back
  int maxit, nrepl;
  int checked;              // the final residual is known
  MgState a, b;
};

// A topology's grids (made once per system, mg_plan).
struct MgPlan {
  bool ok = false;          // false: the rows do not suit one uniform grid
  int n = 0, nlev = 0, tail = 0, steps = 1;
  int nx[MG_MAXLEV], ny[MG_MAXLEV], px[MG_MAXLEV], pn[MG_MAXLEV];
  DevBuf<int> cell, cptr, crow, pos;
  DevBuf<float2> frac, cfrac;
};

// The system's plan (built on the first call); null when the solver should
// not be used for it.
const MgPlan *mg_plan(System &s, hipStream_t st);

// Device floats of the grid levels of one system, and the level pointers of
// a descriptor laid out from `base`.
// (and the partials' pointers, into 5 nblk + 6 doubles: nblk blocks, summed by
// one block or not)
void mg_parts(MgSys &d, int nblk, bool reduce, double *part);
size_t mg_grid_floats(const MgPlan &pl);
void mg_grid_layout(const MgPlan &pl, float *base, MgSys &d);

// Allows the tail kernel the LDS it needs for this plan; how much that is.
void mg_allow_lds(const MgPlan &pl);
size_t mg_tail_lds(const MgPlan &pl);
size_t mg_setup_lds(const MgPlan &pl);

// A batch of systems (descriptors of D, states of S by slot): the block maps
// of every kind of wide launch ((slot, block) per grid block), and the slots.
enum { MGS_ROWS = 0, MGS_TWO, MGS_GALERKIN, MGS_RESTRICT, MGS_SETUP,
       MGS_DOWN = MGS_SETUP + MG_MAXLEV, MGS_UP = MGS_DOWN + MG_MAXLEV,
       MG_STAGES = MGS_UP + MG_MAXLEV };
struct MgBatch {
  int nsys = 0, tail = 0;   // systems; most grids above the tail
  bool reduce = false;      // some system's partials are summed by one block
  size_t tail_lds = 0, setup_lds = 0;
  const int *list = nullptr;
  const int2 *map[MG_STAGES] = {};
  int nmap[MG_STAGES] = {};
};
// the blocks of one system in each of them
void mg_stages(const MgPlan &pl, int npad, int (&nblk)[MG_STAGES]);
void mg_batch_setup(const MgBatch &B, const MgSys *D, hipStream_t st);
void mg_batch_start(const MgBatch &B, const MgSys *D, MgScal *S, double rtol2, int maxit,
                    hipStream_t st);
// iterations, then the check of the systems that stopped; host: pinned copy
// of the states by slot
void mg_batch_iterations(const MgBatch &B, const MgSys *D, MgScal *S, int iters, MgScal *host,
                         hipStream_t st);

}  // namespace admfem
