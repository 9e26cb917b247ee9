// The vertex levels of the multigrid preconditioner on structured meshes.
//
// Level 0 is the reduced trace space (hdg_quad.hip).  Level 1 is the vertex
// space: the prolongation maps vertex values to the Legendre modes 0 and 1 of
// the trace of the linear function on every axis face (mode 0 = mean, mode 1
// = (v_hi - v_lo) / (2 sqrt 3), the face parameter running from the lower to
// the higher node id), and the operator is the Galerkin product P^T T P,
// assembled quad by quad (q_build_kernel, q_l1_kernel).  Levels 2.. are the
// vertex grids coarsened by two (a side with n cells gets (n + 1) / 2: coarse
// node I sits on fine node min(2I, n), so an odd side keeps its last fine
// column as a one-cell-wide coarse column), with bilinear interpolation and
// Galerkin (RAP) operators; every level is a 9-point stencil.  One symmetric
// V-cycle (one damped Jacobi sweep before and after, the coarsest grid
// exactly) is a fixed SPD operator, so it preconditions CG.
//
// Stencil slots: 0 (0,0), 1 (+1,0), 2 (-1,0), 3 (0,+1), 4 (0,-1), 5 (+1,-1),
// 6 (-1,+1), 7 (+1,+1), 8 (-1,-1); node (i, j) of a level with nx cells per
// row is i + j (nx+1).
#include <hip/hip_runtime.h>

#include "hdg_quad.h"

namespace hdg {

namespace {

__constant__ int kOffX[kStencil] = {0, 1, -1, 0, 0, 1, -1, 1, -1};
__constant__ int kOffY[kStencil] = {0, 0, 0, 1, -1, -1, 1, 1, -1};
// slot of offset (dx, dy) at (dy + 1) 3 + dx + 1
__device__ constexpr int kSlotOf[9] = {8, 4, 5, 2, 0, 1, 6, 3, 7};
constexpr int kRapThreads = 64;  // a wavefront per block: the small levels spread over the CUs

// fine index of coarse index I on a side of n fine cells
__device__ __forceinline__ int fine_of(int I, int n) { return min(2 * I, n); }
// weight of coarse index I at fine index x on a side of n fine cells: x even
// or the last node of an odd side has one parent, odd x < n two at 1/2
__device__ __forceinline__ double pw1(int x, int n, int I) {
  if (!(x & 1)) return I == (x >> 1) ? 1.0 : 0.0;
  if (x == n) return I == ((n + 1) >> 1) ? 1.0 : 0.0;
  return I == ((x - 1) >> 1) || I == ((x + 1) >> 1) ? 0.5 : 0.0;
}

// Bilinear interpolation of the coarse vector ec (row length cnx + 1) at fine
// node (x, y) of a level with fnx x fny cells.  (The level-1 operator couples
// the four vertices of a grid cell alike; interpolating along one diagonal
// only costs 3-5 CG iterations: P3 160^2 18 instead of 15.)
__device__ __forceinline__ double prolong_at(int fnx, int fny, int cnx, const double* ec, int x, int y) {
  const int xa = x == fnx ? (fnx + 1) >> 1 : x >> 1, xb = (x & 1) && x != fnx ? xa + 1 : xa;
  const int ya = y == fny ? (fny + 1) >> 1 : y >> 1, yb = (y & 1) && y != fny ? ya + 1 : ya;
  const int64_t cs = cnx + 1;
  return 0.25 * ((ec[ya * cs + xa] + ec[ya * cs + xb]) + (ec[yb * cs + xa] + ec[yb * cs + xb]));
}

// (r, r) <= rtol2 (b, b), the next product's convergence test, taken by the
// first vertex kernel after the update so that a converged solve skips its
// last V-cycle: every block sums the partials in the same order and decides
// alike, the lead block records the state.  rr_part leaves the wavefronts'
// sums in sh; after the caller's next barrier, converged decides.  maxit < 0:
// no test.
__device__ __forceinline__ void rr_part(const double* part, int n, int maxit, double* sh) {
  if (maxit < 0) return;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) s += part[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
}
template <int NW>
__device__ __forceinline__ bool converged(CgState* st, double rtol2, int maxit, bool lead, const double* sh) {
  if (maxit < 0) return false;
  double rr = 0.0;
#pragma unroll
  for (int w = 0; w < NW; ++w) rr += sh[w];
  const int it = st->i_pre;
  const bool conv = rr <= rtol2 * st->bb, stop = conv || it >= maxit;
  if (lead && threadIdx.x == 0) {
    st->it = it;
    st->rr = rr;
    if (stop) st->done = conv ? 1 : 2;
  }
  return stop;
}

// ------------------------------------------------------------ set-up
// Galerkin stencils R A P, R = P^T, a thread per coarse node C: the stencils of
// its support's fine nodes, three at a time, weighted and summed by the node
// they meet, then interpolated, first in x, then in y.  Consecutive threads
// read every other column of a row, so the fine stencils leave HBM once; the
// small levels are bound by two dependent loads.  With 16 lanes per coarse
// node, each spreading one fine node's stencil, and a shuffle tree over the
// lanes: all levels of 1024^2 980 us, now 417 (beside the Lanczos steps), of
// 768^2 288, now 132, a 17 x 17 level 10, now 6.
template <class VS>
__global__ __launch_bounds__(kRapThreads) void mg_rap_kernel(VS sel) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int64_t C = (int64_t)lb * kRapThreads + threadIdx.x;
  if (C >= Cc.n) return;
  constexpr int ox[kStencil] = {0, 1, -1, 0, 0, 1, -1, 1, -1}, oy[kStencil] = {0, 0, 0, 1, -1, -1, 1, 1, -1};
  const int cnx = Cc.nx, cny = Cc.ny, fnx = F.nx, fny = F.ny, row = fnx + 1;
  const int I = (int)(C % (cnx + 1)), J = (int)(C / (cnx + 1)), fx = fine_of(I, fnx), fy = fine_of(J, fny);
  const int64_t f0 = (int64_t)fy * row + fx;
  // fine nodes that are fixed or off the grid
  unsigned off = 0;
#pragma unroll
  for (int p = 0; p < 25; ++p) {
    const int x = fx + p % 5 - 2, y = fy + p / 5 - 2;
    const bool on = x >= 0 && x <= fnx && y >= 0 && y <= fny;
    const unsigned char m = F.mask[on ? (int64_t)y * row + x : f0];
    if (!on || m) off |= 1u << p;
  }
  // own weight at the fine nodes beside C's, per side; their other parent has
  // the rest (an odd side's last node is a parent of its own)
  const double lx = fx & 1 ? 0.0 : 0.5, rx = fx + 1 == fnx ? 0.0 : 0.5;
  const double ly = fy & 1 ? 0.0 : 0.5, ry = fy + 1 == fny ? 0.0 : 0.5;
  double st[kStencil];
#pragma unroll
  for (int k = 0; k < kStencil; ++k) st[k] = 0.0;
  // byte offset of the support's centre (a level has fewer than 2^29 nodes)
  unsigned f1 = 8u * (unsigned)f0;
#pragma unroll
  for (int y = -1; y <= 1; ++y) {
    // the next row's loads wait for this one's sums (all at once take 254
    // registers, and the blocks then wait for room beside the kernels of other
    // streams: up to 440 us in a batch)
    if (y >= 0) asm("" : "+v"(f1), "+v"(st[0]));
    double t[3][5];
#pragma unroll
    for (int k = 0; k < 15; ++k) t[k / 5][k % 5] = 0.0;
#pragma unroll
    for (int x = -1; x <= 1; ++x) {
      const bool use = !((off >> ((y + 2) * 5 + x + 2)) & 1);
      const unsigned fi = use ? f1 + 8u * (unsigned)(y * row + x) : f1;
      const double w = use ? (x == 0 ? 1.0 : (x < 0 ? lx : rx)) * (y == 0 ? 1.0 : (y < 0 ? ly : ry)) : 0.0;
#pragma unroll
      for (int s = 0; s < kStencil; ++s) {
        double& v = t[oy[s] + 1][x + ox[s] + 2];
        v = fma(w, *reinterpret_cast<const double*>(reinterpret_cast<const char*>(F.a + s * F.n) + fi), v);
      }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int py = y + q + 1;
      double v[5];
#pragma unroll
      for (int px = 0; px < 5; ++px) v[px] = (off >> (py * 5 + px)) & 1 ? 0.0 : t[q][px];
      const double u[3] = {fma(1.0 - lx, v[1], v[0]), fma(lx, v[1], fma(rx, v[3], v[2])), fma(1.0 - rx, v[3], v[4])};
      // parents in y: below C's row, C's, above
      const double wy[3] = {py == 0 ? 1.0 : (py == 1 ? 1.0 - ly : 0.0), py == 1 ? ly : (py == 2 ? 1.0 : ry),
                            py == 4 ? 1.0 : (py == 3 ? 1.0 - ry : 0.0)};
#pragma unroll
      for (int dy = 0; dy < 3; ++dy) {
        if ((dy == 0 && py > 1) || (dy == 1 && (py == 0 || py == 4)) || (dy == 2 && py < 3)) continue;
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) st[kSlotOf[dy * 3 + dx]] = fma(wy[dy], u[dx], st[kSlotOf[dy * 3 + dx]]);
      }
    }
  }
  const bool cm = (off >> 12) & 1;
#pragma unroll
  for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
    for (int dx = -1; dx <= 1; ++dx) {
      const int u = kSlotOf[(dy + 1) * 3 + dx + 1], i = I + dx, j = J + dy;
      // columns of fixed coarse nodes are zero; fixed rows are the identity
      const bool in = i >= 0 && i <= cnx && j >= 0 && j <= cny;
      const int p = in ? (fine_of(j, fny) - fy + 2) * 5 + fine_of(i, fnx) - fx + 2 : 12;
      Cc.a[u * Cc.n + C] = cm ? (u == 0 ? 1.0 : 0.0) : (!in || ((off >> p) & 1) ? 0.0 : st[u]);
    }
  Cc.dinv[C] = cm ? 0.0 : 1.0 / st[0];
  Cc.mask[C] = cm ? 1 : 0;
}

// Inverse of the coarsest operator (at most kCoarseDirect nodes), one
// workgroup per hierarchy: in-place Gauss-Jordan without pivoting (the
// operator is SPD, fixed nodes have identity rows; without any fixed node it is
// singular, see kNoPivot), the matrix in registers
// (6 x 6 entries per thread), the pivot row and column through alternating
// LDS buffers, one barrier of four wavefronts per step.  With the pivot p, the
// row and column k take the same fma(-c, r, m) as the rest: the row's factor c
// is p - 1, the column's r is 1 + 1/p (m - (p - 1) m/p = m/p, c - c (1 + 1/p)
// = -c/p).  Bound by the chain of barrier, division and LDS.  With the pivot's
// registers chosen at run time a step took 1.1 us (81 nodes: 88 us, now 42).
__global__ __launch_bounds__(256) void mg_inverse_kernel(const MgData* __restrict__ Ms) {
  constexpr int T = 16, E = kCoarseDirect / T;
  __shared__ double rowb[2][kCoarseDirect], colb[2][kCoarseDirect], mean[kCoarseDirect + 1];
  __shared__ int fixed, dropped;
  const MgData& M = Ms[blockIdx.x];
  const MgLevel& L = M.lev[M.nlev - 1];
  const int n = (int)L.n, tr = threadIdx.x / T, tc = threadIdx.x % T, row = L.nx + 1;
  if (threadIdx.x == 0) fixed = dropped = 0;
  __syncthreads();
  if ((int)threadIdx.x < n && L.mask[threadIdx.x]) fixed = 1;
  double m[E][E], least[E];  // the entries, and the least pivots of those on the diagonal
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int b = 0; b < E; ++b) {
      const int r = tr + T * a, c = tc + T * b;
      double v = 0.0;
      if (r < n && c < n) {
        const int dx = c % row - r % row, dy = c / row - r / row;
        if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1) v = L.a[kSlotOf[(dy + 1) * 3 + dx + 1] * n + r];
      }
      m[a][b] = v;
    }
#pragma unroll
  for (int a = 0; a < E; ++a) least[a] = tr == tc ? kNoPivot * m[a][a] : -1.0;
  // k = ka T + kt with ka unrolled, so that the pivot's registers are known
#pragma unroll
  for (int ka = 0; ka < E; ++ka)
    for (int kt = 0; kt < T && ka * T + kt < n; ++kt) {
      const int k = ka * T + kt, p = kt & 1;
      const bool none = tc == kt && fabs(m[ka][ka]) <= least[ka];
      if (none) dropped = 1;
      if (tr == kt)
#pragma unroll
        for (int b = 0; b < E; ++b) rowb[p][tc + T * b] = b == ka && none ? kLeftOut : m[ka][b];
      if (tc == kt)
#pragma unroll
        for (int a = 0; a < E; ++a) colb[p][tr + T * a] = m[a][ka];
      __syncthreads();
      const double piv = rowb[p][k];
      double rk[E], ck[E];
#pragma unroll
      for (int a = 0; a < E; ++a) {
        rk[a] = rowb[p][tc + T * a];
        ck[a] = colb[p][tr + T * a];
      }
      const double ip = 1.0 / piv;
#pragma unroll
      for (int a = 0; a < E; ++a) rk[a] *= ip;
      rk[ka] = tc == kt ? 1.0 + ip : rk[ka];
      ck[ka] = tr == kt ? piv - 1.0 : ck[ka];
#pragma unroll
      for (int a = 0; a < E; ++a)
#pragma unroll
        for (int b = 0; b < E; ++b) m[a][b] = fma(-ck[a], rk[b], m[a][b]);
      m[ka][ka] = none ? 0.0 : m[ka][ka];
    }
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int b = 0; b < E; ++b) {
      const int r = tr + T * a, c = tc + T * b;
      if (r < n && c < n) M.cinv[r * n + c] = m[a][b];
    }
  if (dropped && !fixed) project_constants(M.cinv, n, mean);
}

// ------------------------------------------------------- vertex levels
// The level kernels take a selector (VOne, VGroup) that names the instance of
// the block: its fine level F, coarse level C and CG state.  Both stage in
// LDS what neighbouring nodes share, so that a node's stencil, right-hand side
// and inverse diagonal are read once: HBM-bound on the finest level (11
// doubles per node), launch latency below.

// coarse r = R (r - A e), R = P^T, e = om dinv r the pre-smoothing sweep from
// zero: a block owns kRX x kRY coarse nodes and forms the residuals of their
// (2 kRX + 1) x (2 kRY + 1) fine nodes once.  (Eight lanes per coarse node,
// each forming the residuals it needs, 2.25 per fine node: 1024^2 P3 75 us
// per V-cycle over all levels; now 64, at 512^2 26.)
constexpr int kRX = 16, kRY = 8;
template <class VS>
__global__ __launch_bounds__(256) void v_restrict_kernel(VS sel, double om, double rtol2, int maxit) {
  constexpr int WX = 2 * kRX + 1, WY = 2 * kRY + 1, EX = WX + 2, EY = WY + 2;
  __shared__ double e[EY * EX], d[WY * WX], sh[4];
  constexpr int NE = (EX * EY + 255) / 256, ND = (WX * WY + 255) / 256;
  int lb;
  const VRec& R = vrec_of(sel, lb);
  const int done = R.st->done;
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int ntx = Cc.nx / kRX + 1;
  const int I0 = (lb % ntx) * kRX, J0 = (lb / ntx) * kRY, x0 = 2 * I0 - 1, y0 = 2 * J0 - 1;
  const int row = F.nx + 1;
  // every load before the first barrier: the sweep's factors on the tile and
  // its border, the stencils of the tile's nodes
  double ev[NE], av[ND][kStencil], rv[ND];
  bool fr[ND];
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    const int u = threadIdx.x + 256 * k, x = x0 - 1 + u % EX, y = y0 - 1 + u / EX;
    const bool on = u < EX * EY && x >= 0 && x <= F.nx && y >= 0 && y <= F.ny;
    const int64_t g = on ? (int64_t)y * row + x : 0;
    const double v = om * F.dinv[g] * F.r[g];
    ev[k] = on ? v : 0.0;
  }
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    const int u = threadIdx.x + 256 * k, x = x0 + u % WX, y = y0 + u / WX;
    const bool on = u < WX * WY && x >= 0 && x <= F.nx && y >= 0 && y <= F.ny;
    const int64_t g = on ? (int64_t)y * row + x : 0;
#pragma unroll
    for (int s = 0; s < kStencil; ++s) av[k][s] = F.a[s * F.n + g];
    rv[k] = F.r[g];
    fr[k] = on && F.dinv[g] != 0.0;
  }
  if (done) return;
  rr_part(R.part, R.npart, maxit, sh);
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    const int u = threadIdx.x + 256 * k;
    if (u < EX * EY) e[u] = ev[k];
  }
  __syncthreads();
  if (converged<4>(R.st, rtol2, maxit, lb == 0, sh)) return;
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    const int u = threadIdx.x + 256 * k;
    if (u < WX * WY) {
      const double* ep = e + (u / WX + 1) * EX + u % WX + 1;
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < kStencil; ++q) s = fma(av[k][q], ep[kOffY[q] * EX + kOffX[q]], s);
      d[u] = fr[k] ? rv[k] - s : 0.0;
    }
  }
  __syncthreads();
  if (threadIdx.x >= kRX * kRY) return;
  const int I = I0 + (int)threadIdx.x % kRX, J = J0 + (int)threadIdx.x / kRX;
  if (I > Cc.nx || J > Cc.ny) return;
  const int fx = fine_of(I, F.nx), fy = fine_of(J, F.ny);
  double s = 0.0;
#pragma unroll
  for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
    for (int dx = -1; dx <= 1; ++dx) {
      const double w = pw1(fx + dx, F.nx, I) * pw1(fy + dy, F.ny, J);
      if (w != 0.0) s = fma(w, d[(fy + dy - y0) * WX + fx + dx - x0], s);
    }
  const int64_t C = (int64_t)J * (Cc.nx + 1) + I;
  Cc.r[C] = Cc.mask[C] ? 0.0 : s;
}

// e = e' + om dinv (r - A e'), e' = om dinv r + P ec on free nodes: the
// prolongation and the post-smoothing sweep, a block owning kPX x kPY nodes
// (37 us per V-cycle over all levels at 1024^2; 64 us with the prolongation
// repeated at every neighbour that reads it).
constexpr int kPX = 32, kPY = 8;
template <class VS>
__global__ __launch_bounds__(256) void v_post_kernel(VS sel, double om) {
  constexpr int EX = kPX + 2, EY = kPY + 2;
  __shared__ double e[EY * EX];
  int lb;
  const VRec& R = vrec_of(sel, lb);
  const int done = R.st->done;
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int ntx = F.nx / kPX + 1;
  const int x0 = (lb % ntx) * kPX, y0 = (lb / ntx) * kPY, row = F.nx + 1;
  const int wx = threadIdx.x % kPX, wy = threadIdx.x / kPX;
  const bool own = x0 + wx <= F.nx && y0 + wy <= F.ny;
  const int64_t g = own ? (int64_t)(y0 + wy) * row + x0 + wx : 0;
  double av[kStencil];
#pragma unroll
  for (int q = 0; q < kStencil; ++q) av[q] = F.a[q * F.n + g];
  const double rv = F.r[g], di = F.dinv[g];
  // the tile and its border, loaded with the stencils ahead of the branch
  constexpr int NE = (EX * EY + 255) / 256;
  double ev[NE];
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    const int u = threadIdx.x + 256 * k, x = x0 - 1 + u % EX, y = y0 - 1 + u / EX;
    const bool on = u < EX * EY && x >= 0 && x <= F.nx && y >= 0 && y <= F.ny;
    const int xc = on ? x : 0, yc = on ? y : 0;
    const int64_t gg = (int64_t)yc * row + xc;
    const double dd = F.dinv[gg], p = prolong_at(F.nx, F.ny, Cc.nx, Cc.e, xc, yc);
    ev[k] = on && dd != 0.0 ? fma(om * dd, F.r[gg], p) : 0.0;
  }
  if (done) return;
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    const int u = threadIdx.x + 256 * k;
    if (u < EX * EY) e[u] = ev[k];
  }
  __syncthreads();
  if (!own) return;
  const double* ep = e + (wy + 1) * EX + wx + 1;
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < kStencil; ++q) s = fma(av[q], ep[kOffY[q] * EX + kOffX[q]], s);
  F.e[g] = fma(om * di, rv - s, ep[0]);
}

// Levels tail .. nlev-1 of the V-cycle in one workgroup per hierarchy (Ms[b]
// with CG state sts[b]): reads lev[tail].r, writes lev[tail].e.  The levels'
// nodes (at most kTailNodes) are laid end to end, two per thread, whose
// stencils, inverse diagonals and the LDS positions of what they read stay in
// registers; the vectors that neighbours read are in LDS.  A neighbour off the
// grid is read at the nearest node on it, with a zero coefficient.  Bound by
// its chain of phases: two per level down (the residual, the restriction), one
// for the coarsest grid, two per level up; every load comes before the first.
// 33 x 33: 11.9 us, 17.4 with the positions and weights worked out in every
// phase.
__global__ __launch_bounds__(kTailThreads) void v_tail_kernel(const MgData* __restrict__ Ms, CgState* sts, double rtol2,
                                                              int maxit) {
  constexpr int Q = (kTailNodes + kTailThreads - 1) / kTailThreads, NI = kCoarseDirect / 8;
  static_assert(8 * kCoarseDirect <= kTailThreads, "eight lanes per row of the coarsest inverse");
  __shared__ double Z[kTailNodes], Y[kTailNodes], X[kTailNodes];
  __shared__ double sh[kTailThreads / 64];
  const MgData& M = Ms[blockIdx.x];
  CgState* st = sts + blockIdx.x;
  const int done = st->done;
  const double om = M.omega_v;
  const int lt = M.tail, last = M.nlev - 1, tid = threadIdx.x;
  // own nodes: level; position in the vectors (v), of the fine node under it
  // (f) and of the coarse node at its lower left (pa); flags: neighbours on
  // the grid (kL ..), restriction weights that are 1/2 (kFl ..), whether it
  // lies between coarse columns (kPx) or rows (kPy)
  enum { kL = 1, kR = 2, kD = 4, kU = 8, kFl = 16, kFr = 32, kFd = 64, kFu = 128, kPx = 256, kPy = 512 };
  int lev[Q], v[Q], f[Q], pa[Q], fg[Q];
  double a[Q][kStencil], di[Q], r[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    lev[q] = -1;
    v[q] = f[q] = pa[q] = fg[q] = 0;
    di[q] = r[q] = 0.0;
#pragma unroll
    for (int k = 0; k < kStencil; ++k) a[q][k] = 0.0;
  }
  // level by level, so that sizes and pointers are the wavefront's
  for (int l = lt, o = 0, op = 0; l <= last; ++l) {
    const MgLevel& L = M.lev[l];
    const int nx = L.nx, ny = L.ny, row = nx + 1, n = (int)L.n;
    const int fnx = l > lt ? M.lev[l - 1].nx : 0, fny = l > lt ? M.lev[l - 1].ny : 0;
    const int cs = l < last ? M.lev[l + 1].nx + 1 : 0;
    const double *La = L.a, *Ld = L.dinv, *Lr = L.r;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int u = tid + q * kTailThreads - o;
      if (u < 0 || u >= n) continue;
#pragma unroll
      for (int k = 0; k < kStencil; ++k) a[q][k] = La[k * n + u];
      di[q] = om * Ld[u];
      if (l == lt) r[q] = Lr[u];
      const int x = u % row, y = u / row;
      lev[q] = l;
      v[q] = o + u;
      int g = (x > 0 ? kL : 0) | (x < nx ? kR : 0) | (y > 0 ? kD : 0) | (y < ny ? kU : 0);
      if (l > lt) {
        const int fx = fine_of(x, fnx), fy = fine_of(y, fny);
        f[q] = op + fy * (fnx + 1) + fx;
        if (fx > 0 && pw1(fx - 1, fnx, x) != 0.0) g |= kFl;
        if (fx < fnx && pw1(fx + 1, fnx, x) != 0.0) g |= kFr;
        if (fy > 0 && pw1(fy - 1, fny, y) != 0.0) g |= kFd;
        if (fy < fny && pw1(fy + 1, fny, y) != 0.0) g |= kFu;
      }
      if (l < last) {
        const int xa = x == nx ? (nx + 1) >> 1 : x >> 1, ya = y == ny ? (ny + 1) >> 1 : y >> 1;
        pa[q] = o + n + ya * cs + xa;
        if ((x & 1) && x != nx) g |= kPx;
        if ((y & 1) && y != ny) g |= kPy;
      }
      fg[q] = g;
    }
    op = o;
    o += n;
  }
  double ci[NI];
  const int nc = (int)M.lev[last].n, cv = tid >> 3, ct = tid & 7;
#pragma unroll
  for (int k = 0; k < NI; ++k) {
    const int u = ct + 8 * k;
    ci[k] = cv < nc && u < nc ? M.cinv[cv * nc + u] : 0.0;
  }
  if (done) return;
  if (lt == 1) rr_part(M.part, M.npart, maxit, sh);
  // slots with a neighbour off the grid: to the right 1, 5, 7, left 2, 6, 8,
  // above 3, 6, 7, below 4, 5, 8
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const bool xl = fg[q] & kL, xr = fg[q] & kR, yd = fg[q] & kD, yu = fg[q] & kU;
    a[q][1] = xr ? a[q][1] : 0.0;
    a[q][2] = xl ? a[q][2] : 0.0;
    a[q][3] = yu ? a[q][3] : 0.0;
    a[q][4] = yd ? a[q][4] : 0.0;
    a[q][5] = xr && yd ? a[q][5] : 0.0;
    a[q][6] = xl && yu ? a[q][6] : 0.0;
    a[q][7] = xr && yu ? a[q][7] : 0.0;
    a[q][8] = xl && yd ? a[q][8] : 0.0;
  }
  const auto stencil = [&](int q, const double* W, int row) {
    const int c = v[q], m = c - (fg[q] & kD ? row : 0), p = c + (fg[q] & kU ? row : 0);
    const int lft = fg[q] & kL ? -1 : 0, rgt = fg[q] & kR ? 1 : 0;
    double s = a[q][0] * W[c];
    s = fma(a[q][1], W[c + rgt], s);
    s = fma(a[q][2], W[c + lft], s);
    s = fma(a[q][3], W[p], s);
    s = fma(a[q][4], W[m], s);
    s = fma(a[q][5], W[m + rgt], s);
    s = fma(a[q][6], W[p + lft], s);
    s = fma(a[q][7], W[p + rgt], s);
    return fma(a[q][8], W[m + lft], s);
  };
  int o = 0;
  for (int l = lt; l < last; ++l) {
    const int row = M.lev[l].nx + 1;
    // the sweep from zero
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (lev[q] == l) Z[v[q]] = di[q] * r[q];
    __syncthreads();
    if (l == 1 && converged<kTailThreads / 64>(st, rtol2, maxit, true, sh)) return;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (lev[q] == l) Y[v[q]] = di[q] == 0.0 ? 0.0 : r[q] - stencil(q, Z, row);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (lev[q] == l + 1) {
        // a fine neighbour of weight zero is read at the node itself
        const int g = fg[q], c = f[q], m = c - (g & kFd ? row : 0), p = c + (g & kFu ? row : 0);
        const int lft = g & kFl ? -1 : 0, rgt = g & kFr ? 1 : 0;
        const double wl = g & kFl ? 0.5 : 0.0, wr = g & kFr ? 0.5 : 0.0;
        const double s0 = fma(wl, Y[c + lft], fma(wr, Y[c + rgt], Y[c]));
        const double sm = fma(wl, Y[m + lft], fma(wr, Y[m + rgt], Y[m]));
        const double sp = fma(wl, Y[p + lft], fma(wr, Y[p + rgt], Y[p]));
        const double s = fma(g & kFd ? 0.5 : 0.0, sm, fma(g & kFu ? 0.5 : 0.0, sp, s0));
        r[q] = di[q] == 0.0 ? 0.0 : s;
        if (l + 1 == last) Z[v[q]] = r[q];
      }
    o += (int)M.lev[l].n;
  }
  if (lt == last) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (lev[q] == last) Z[v[q]] = r[q];
  }
  __syncthreads();
  if (lt == last && lt == 1 && converged<kTailThreads / 64>(st, rtol2, maxit, true, sh)) return;
  {
    // coarsest grid: eight lanes per row of its inverse
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int u = ct + 8 * k;
      s = fma(ci[k], Z[o + (u < nc ? u : 0)], s);
    }
    s += __shfl_xor(s, 1, 8);
    s += __shfl_xor(s, 2, 8);
    s += __shfl_xor(s, 4, 8);
    if (cv < nc && ct == 0) X[o + cv] = s;
    __syncthreads();
  }
  for (int l = last - 1; l >= lt; --l) {
    const int row = M.lev[l].nx + 1, cs = M.lev[l + 1].nx + 1;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (lev[q] == l) {
        const double* e = X + pa[q];
        const int dx = fg[q] & kPx ? 1 : 0, dy = fg[q] & kPy ? cs : 0;
        const double p = 0.25 * ((e[0] + e[dx]) + (e[dy] + e[dy + dx]));
        Y[v[q]] = di[q] == 0.0 ? 0.0 : fma(di[q], r[q], p);
      }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (lev[q] == l) {
        const double ev = fma(di[q], r[q] - stencil(q, Y, row), Y[v[q]]);
        X[v[q]] = ev;
        if (l == lt) M.lev[lt].e[v[q]] = ev;
      }
    if (l > lt) __syncthreads();
  }
  if (lt == last && cv < nc && ct == 0) M.lev[lt].e[cv] = X[cv];
}

}  // namespace

int v_rap_blocks(const MgLevel& C) { return (int)((C.n + kRapThreads - 1) / kRapThreads); }
int v_restrict_blocks(const MgLevel& C) { return (C.nx / kRX + 1) * (C.ny / kRY + 1); }
int v_post_blocks(const MgLevel& F) { return (F.nx / kPX + 1) * (F.ny / kPY + 1); }

int mg_setup_levels(const MgData& M, const MgData* dM, hipStream_t s) {
  for (int l = 1; l + 1 < M.nlev; ++l) {
    const VOne rec{VRec{M.lev[l], M.lev[l + 1], nullptr, nullptr, 0}};
    hipLaunchKernelGGL(mg_rap_kernel<VOne>, dim3(v_rap_blocks(M.lev[l + 1])), dim3(kRapThreads), 0, s, rec);
  }
  hipLaunchKernelGGL(mg_inverse_kernel, dim3(1), dim3(256), 0, s, dM);
  return (int)hipGetLastError();
}

int mg_setup_levels_group(const MgSetupGroup& S, hipStream_t s) {
  for (int d = 1; d < S.ndepth; ++d)
    hipLaunchKernelGGL(mg_rap_kernel<VGroup>, dim3(S.grap[d]), dim3(kRapThreads), 0, s, S.rap[d]);
  hipLaunchKernelGGL(mg_inverse_kernel, dim3(S.ninst), dim3(256), 0, s, S.dM);
  return (int)hipGetLastError();
}

int launch_vcycle(const MgData& M, const MgData* dM, CgState* st, double rtol2, int maxit, hipStream_t s) {
  for (int l = 1; l < M.tail; ++l) {
    const VOne rec{VRec{M.lev[l], M.lev[l + 1], st, M.part, M.npart}};
    hipLaunchKernelGGL(v_restrict_kernel<VOne>, dim3(v_restrict_blocks(M.lev[l + 1])), dim3(256), 0, s, rec, M.omega_v,
                       rtol2, l == 1 ? maxit : -1);
  }
  hipLaunchKernelGGL(v_tail_kernel, dim3(1), dim3(kTailThreads), 0, s, dM, st, rtol2, maxit);
  for (int l = M.tail - 1; l >= 1; --l) {
    const VOne rec{VRec{M.lev[l], M.lev[l + 1], st, nullptr, 0}};
    hipLaunchKernelGGL(v_post_kernel<VOne>, dim3(v_post_blocks(M.lev[l])), dim3(256), 0, s, rec, M.omega_v);
  }
  return (int)hipGetLastError();
}

// The same V-cycle for every instance of a group: depth by depth down to the
// tails, every tail in one launch (one workgroup each), depth by depth up.
// An instance whose tail starts at depth t takes part in depths 1..t-1 only.
int launch_vcycle_group(const MgGroup& G, double rtol2, int maxit, hipStream_t s) {
  for (int d = 1; d < G.ndepth; ++d)
    hipLaunchKernelGGL(v_restrict_kernel<VGroup>, dim3(G.gres[d]), dim3(256), 0, s, G.res[d], G.omega_v, rtol2,
                       d == 1 ? maxit : -1);
  hipLaunchKernelGGL(v_tail_kernel, dim3(G.ninst), dim3(kTailThreads), 0, s, G.dM, G.st, rtol2, maxit);
  for (int d = G.ndepth - 1; d >= 1; --d)
    hipLaunchKernelGGL(v_post_kernel<VGroup>, dim3(G.gnode[d]), dim3(256), 0, s, G.node[d], G.omega_v);
  return (int)hipGetLastError();
}

}  // namespace hdg
