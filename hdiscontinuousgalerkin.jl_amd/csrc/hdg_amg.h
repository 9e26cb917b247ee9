// Multigrid preconditioner of the trace CG on meshes without rectangle
// structure: block-Jacobi on the trace, the continuous linear functions on
// the mesh's vertices, smoothed aggregation below them.
//
// With J = Dinv, S = -K and P the map from vertex values to face modes 0 and
// 1 (the trace of the linear function: mean, (v_hi - v_lo) / (2 sqrt 3)), one
// V(1,1) cycle from zero is
//   z = (2 w J - w^2 J S J) r + G A^-1 G^T r,   G = (I - w J S) P,
// so a cycle needs one product with S (beside the restriction), and the
// transfer G, formed once per solve, carries both the sweeps' part and the
// interpolation.  The vertex levels have the same form, G_l = (I - w D_l A_l)
// P_l.  w J and w D are small enough for an SPD cycle whatever the mesh: S is
// a sum over cells of semidefinite blocks of three faces, so J S <= 3 and w =
// 0.6 < 2/3; D_l = 1 / max(a_ii, half the row's absolute sum), so D_l A_l <= 2
// and 0.8 < 1.
#pragma once
#include <vector>

#include "hdg_internal.h"

namespace hdg {

constexpr double kAmgOmega = 0.6, kAmgOmegaV = 0.8, kAmgOmegaP = 2.0 / 3.0;
constexpr int kAmgLevels = 16;
// coarsening stops at this many nodes, solved by the operator's inverse
constexpr int kAmgDirect = 96;
// the last levels' cycle is formed as one matrix: its rows (8 MB), and the
// nodes of all its levels (vectors in LDS while it is formed)
constexpr int kAmgDense = 1024, kAmgTailNodes = 2048;

// A vertex level: the operator (CSR, rows sorted) and, but for the last
// level, the transfer to the next one by rows (gp, gi, gv) and by columns
// (tp; row ti of the entry at position tx of gv)
struct AmgLevel {
  int n = 0;
  const int *ap = nullptr, *ai = nullptr, *agg = nullptr;
  const int *gp = nullptr, *gi = nullptr, *tp = nullptr, *ti = nullptr, *tx = nullptr;
  double *av = nullptr, *gv = nullptr;
  double *pv = nullptr, *apv = nullptr;  // P and A P on G's pattern (set-up)
  double *dinv = nullptr;                // kAmgOmegaV D
  double *r = nullptr, *e = nullptr;
};

// The trace space beside level 0: fv[4f + j] = the ends of face f (lower id,
// higher id) and the vertices opposite to it in its cells (or -1); per vertex
// the codes 4f + j that name it; af = the face between the two vertices of an
// entry of level 0's operator (-1 on the diagonal; two entries where the mesh is
// cut open along an edge).  cv = the cells' vertices: their nodes, or, where a
// face joins two edges of the mesh, one node for those it brings together.
struct AmgTop {
  int n = 0;
  const int* cv = nullptr;
  const int *fv = nullptr, *vp = nullptr, *vi = nullptr, *af = nullptr;
  unsigned char* vfix = nullptr;  // vertex of a face with prescribed dofs
  double* g = nullptr;            // G: row r of vertex j at g[j N + r]
  double* t = nullptr;            // the sweeps' part of z
  double *r = nullptr, *e = nullptr;  // level 0's vectors
};

struct AmgData {
  int nlev = 0, tail = 0;
  bool direct = false;  // the last level by its inverse, else one sweep
  AmgLevel lev[kAmgLevels];
  double* cinv = nullptr;
  double* dense = nullptr;  // the cycle of levels tail .. nlev-1 (none: tail = nlev)
  AmgTop top;
};

// The integer arrays of the hierarchy, laid end to end in `ints` (offsets,
// in ints, in the fields of `off`), from the mesh alone.
struct AmgPlan {
  int nlev = 0, tail = 0;
  bool direct = false;
  struct Level {
    int n = 0, nnz = 0, gnnz = 0;
    size_t ap, ai, agg, gp, gi, tp, ti, tx;
  } lev[kAmgLevels];
  size_t fv, vp, vi, af, cv = 0;
  bool joined = false;  // cv is there
  std::vector<int> ints;
};
// The aspect that a quarter of the cells exceed: the square of the longest
// edge over four times the area, 1 for half a square, s / 2 for half a
// rectangle of s by 1.
double amg_aspect(int64_t nc, const int* cn, const double* xy);
// false: the mesh's lists do not fit 32-bit indices, or do not fit together
bool amg_plan(int64_t nn, int64_t nc, int64_t nf, const int* cn, const int* cf, const int* fcell, AmgPlan& plan);

// operators and transfers of the current matrix (T with its Jacobi blocks)
int launch_amg_setup(const DevMesh& m, const TraceSystem& T, const double* Ate, const AmgData& A, const AmgData* dA,
                     hipStream_t s);
// z = the cycle's result for cg.r, given cg.z = J r; the (r, z) partials of
// the next product.  maxit >= 0: takes that product's convergence test first.
int launch_amg_cycle(const DevPattern& P, const TraceSystem& T, const CgVectors& cg, const AmgData& A,
                     double rtol2, int maxit, hipStream_t s);

}  // namespace hdg
