// The trace solve on rectangle meshes (hdg_quad.hip).  Not part of the
// public ABI.
//
// Every grid cell (i, j) of a rectangle_mesh holds two triangles that share
// the diagonal face D; D meets no other cell, so the D blocks of the trace
// system decouple from each other and are eliminated exactly.  What is left
// couples the axis faces: H(i, j) from node (i, j) to (i+1, j) and V(i, j)
// from (i, j) to (i, j+1).  Grid cell ("quad") (i, j) couples B = H(i, j),
// T = H(i, j+1), L = V(i, j) and R = V(i+1, j).  This system has two thirds
// of the unknowns and, preconditioned the same way, takes about half the CG
// iterations of the full one (P3 160^2: 15 instead of 28, P2 25 / 36, P1
// 13 / 26): the coarse functions are extended to the diagonals by the exact
// local solve instead of linearly.
//
// Data live on the grid points g = i + j (nx+1) (point (i, j) carries H(i, j),
// V(i, j), vertex (i, j) and quad (i, j); what does not exist is zero and
// masked), in tiles of 64 points: value s of point g of an array with NS
// values per point is at ((tile0 + g / 64) NS + s) 64 + g % 64, so that a
// wavefront's loads of one value are 64 consecutive doubles and a point's
// values lie in one piece of a few tens of KB.  No index arrays.
#pragma once
#include "hdg_internal.h"

namespace hdg {

// One rectangle problem: its grid, its part of the launches and of the
// packed arrays.
struct QuadInst {
  int nx = 0, ny = 0, W = 0;  // W = nx + 1 points per row
  int G = 0;                  // points
  int ntiles = 0;
  int64_t tile0 = 0;          // first tile in the packed arrays
  int64_t cell0 = 0;          // first triangle in the packed mesh
  // the marching kernels: a block's four wavefronts walk R grid rows each, one
  // above the other; NG groups of 4 R rows, tasks of kQuadOwn columns of the
  // groups laid end to end
  int R = 1, NG = 0, tasks = 0;
  // blocks of the marching and of the pointwise kernels; their first
  // partial sums
  int nbM = 0, nbE = 0, pM = 0, pE = 0;
  int nbQ = 0;  // blocks of the set-up and finish kernels
  CgState* st = nullptr;
  int* plain = nullptr;  // != 0: a diagonal face has prescribed dofs (no constant shift)
  // vertex level 1
  double *r1 = nullptr, *e1 = nullptr;
  double *l1a = nullptr, *l1dinv = nullptr;
  unsigned char* vmask = nullptr;
};
constexpr int kQuadOwn = 62;     // columns a wavefront of a marching kernel owns (64 less two halo lanes)
constexpr int kQuadThreads = 256;
void quad_plan(int nx, int ny, int nt, QuadInst& I);

// the arrays of one or several (packed) problems
struct QuadSys {
  int nt = 0;
  int64_t tiles = 0;
  int nbt = 0;            // partial-sum stride
  int shift = 0;          // tau = 1: the system annihilates constants away from the boundary
  double *blk = nullptr;  // 6 nt^2: BT LR BL BR TL TR, row-major
  double *D = nullptr, *Dinv = nullptr;  // 2 triangles: H, V
  double *tp = nullptr;   // 12 nt: T P on the 6 vertices of H, of V (set-up scratch before)
  double *bq = nullptr;   // 9 nt: per-quad loads (reduced, raw, diagonal)
  double *cq = nullptr;   // 10: per-quad P^T T P
  float *fblk = nullptr, *fDinv = nullptr, *ftp = nullptr;  // HDG_MIXED
  unsigned short* mask = nullptr;  // bits 0..nt-1 H, nt..2nt-1 V
  double *x = nullptr, *r0 = nullptr, *r1 = nullptr, *z = nullptr, *p = nullptr, *q = nullptr, *res = nullptr;
  double* part = nullptr;  // 5 nbt
  const int* cf = nullptr;
  const unsigned char* dmask = nullptr;
  const double* uD = nullptr;
  const double *Ate = nullptr, *bte = nullptr;
  // the assembled matrix, its entries rounded to float as they are read,
  // instead of the cells' blocks (hdg_refine_probe)
  int from_k = 0;
  DevPattern P;
  TraceSystem K;
};
// doubles per point of the arrays above (x .. res: 2 nt each)
__host__ __device__ inline int quad_blk_vals(int nt) { return 6 * nt * nt; }
inline int quad_diag_vals(int nt) { return nt * (nt + 1); }
inline int quad_tp_vals(int nt) { return 12 * nt; }
inline int quad_bq_vals(int nt) { return 9 * nt; }
constexpr int kQuadCq = 10;
constexpr int kQuadVecs = 7;
constexpr int kQuadPartials = 5;

// A launch over one problem (inst null) or over a group: block maps of the
// marching, pointwise and per-quad kernels.
struct QuadLaunch {
  QuadInst one;
  const QuadInst* inst = nullptr;
  const BlockMap *mapM = nullptr, *mapE = nullptr, *mapQ = nullptr;
  int gM = 0, gE = 0, gQ = 0, ninst = 1;
};
QuadLaunch quad_launch_one(const QuadInst& I, int nt);

// once per set-up, before the first launch_quad_build
int launch_quad_clear(const QuadSys& S, const QuadLaunch& L, hipStream_t s);
// masks, the reduced system and its loads from the condensed cells, D, Dinv
int launch_quad_build(const QuadSys& S, const QuadLaunch& L, hipStream_t s);
// float copies for HDG_MIXED (after launch_quad_tp)
int launch_quad_float(const QuadSys& S, hipStream_t s);
// T P, and the stencils of vertex level 1
int launch_quad_tp(const QuadSys& S, const QuadLaunch& L, hipStream_t s);
int launch_quad_l1(const QuadSys& S, const QuadLaunch& L, hipStream_t s);
// the smoothing weight from `steps` Lanczos steps (uses r0, z, p, q)
int launch_quad_omega(const QuadSys& S, const QuadLaunch& L, double factor, int steps, hipStream_t s);
int launch_quad_init(const QuadSys& S, const QuadLaunch& L, hipStream_t s);
// CG product with the convergence test; update and level-0 residual with the
// restriction to the vertices; post-smoothing.  mixed selects the
// preconditioner's storage.
int launch_quad_product(const QuadSys& S, const QuadLaunch& L, double rtol2, int maxit, hipStream_t s);
int launch_quad_residual(const QuadSys& S, const QuadLaunch& L, bool mixed, hipStream_t s);
int launch_quad_smooth(const QuadSys& S, const QuadLaunch& L, bool mixed, hipStream_t s);
// uhat (natural numbering) with the diagonals' solution; with out, also
// ||K uhat - rhs||^2 over the free dofs of every instance
int launch_quad_finish(const QuadSys& S, const QuadLaunch& L, double* uhat, double* out, hipStream_t s);
// one product / update launch regardless of the convergence state, for timing
int launch_quad_time(const QuadSys& S, const QuadLaunch& L, int which, hipStream_t s);

// the smoothing weight over the Lanczos estimate of lambda_max(Dinv T), by
// order
double quad_omega_factor(int k);

// V-cycle on the vertex levels, the next product's convergence test first
// (maxit < 0: none)
int launch_vcycle(const MgData& M, const MgData* dM, CgState* st, double rtol2, int maxit, hipStream_t s);
int launch_vcycle_group(const MgGroup& G, double rtol2, int maxit, hipStream_t s);

}  // namespace hdg
