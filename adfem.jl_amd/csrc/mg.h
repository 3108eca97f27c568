// Multigrid-preconditioned CG for mesh systems (mg.hip): structures shared by
// the single-system solver and the serving engine.
#pragma once
#include "internal.h"

namespace admfem {

constexpr int MG_MAXLEV = 16;    // grid levels at most
constexpr int MG_HALO = 2;       // zero nodes around a grid (the stencils reach 2)
constexpr int MG_TAIL = 2048;    // padded nodes of the first level of the tail kernel
constexpr int MG_DENSE = 64;     // nodes of the last level at most (dense inverse)

// One grid level: nx x ny nodes stored with a halo of MG_HALO zero nodes on
// every side (pitch px, pn entries in all), node (x, y) at mg_at.
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

// One system: its matrix, the plan's arrays (shared by every system of the
// topology) and its vectors (internal row order, npad long).
struct MgSys {
  const int *sp, *sc;       // SELL slice offsets / columns
  const int16_t *sd;        // the columns as 16-bit offsets from the row, or null
  const int *row_bd;
  const double *sv64, *diag;  // FP64 matrix
  float *sv32;              // scaled off-diagonals a_ij / sqrt(a_ii a_jj)
  double *dsq;              // 1 / sqrt(a_ii)
  float *sq, *minv;         // sqrt(a_ii), smoother's weights
  const int *cell;          // grid cell of each row (-1: not interpolated)
  const float2 *frac;       // position inside the cell
  const int *cptr, *crow;   // rows by cell
  const double *b;          // right-hand side
  double *x, *r, *q, *p[2];
  float *z, *rs, *x0, *t;   // preconditioned residual, scaled residual,
                            // smoothed correction, residual / corrected
  double *part;             // 4 x nblk block partials
  float *cinv;              // dense inverse of the last level
  int n, npad, nblk;
  int nlev, tail;           // grid levels, first one of the tail kernel
  MgLevel lv[MG_MAXLEV];
};

struct MgScal {
  double rtol2, bb, tol2, rr, rz, alpha, beta;
  int status;               // as in cg.hip: 0 run, 1 converged, 2 iterations
                            // spent, 3 NaN, 4 breakdown
  int it, maxit, apply, first, nrepl;
};

// A topology's grids (made once per system, mg_plan).
struct MgPlan {
  bool ok = false;          // false: the rows do not suit one uniform grid
  int nlev = 0, tail = 0;
  int nx[MG_MAXLEV], ny[MG_MAXLEV], px[MG_MAXLEV], pn[MG_MAXLEV];
  DevBuf<int> cell, cptr, crow;
  DevBuf<float2> frac;
  size_t bytes() const { return cell.bytes() + cptr.bytes() + crow.bytes() + frac.bytes(); }
};

// The system's plan (built on the first call); null when the solver should
// not be used for it.
const MgPlan *mg_plan(System &s, hipStream_t st);

// Device floats of the grid levels of one system, and the level pointers of
// a descriptor laid out from `base`.
size_t mg_grid_floats(const MgPlan &pl);
void mg_grid_layout(const MgPlan &pl, float *base, MgSys &d);

}  // namespace admfem
