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
// V-cycle (damped Jacobi, fixed sweep counts, the coarsest grid exactly or by
// Jacobi sweeps) is a fixed SPD operator, so it preconditions CG.
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

__device__ inline int slot_of(int dx, int dy) {
  if (dx == 0 && dy == 0) return 0;
  if (dy == 0) return dx == 1 ? 1 : (dx == -1 ? 2 : -1);
  if (dx == 0) return dy == 1 ? 3 : (dy == -1 ? 4 : -1);
  if (dx == 1 && dy == -1) return 5;
  if (dx == -1 && dy == 1) return 6;
  if (dx == 1 && dy == 1) return 7;
  if (dx == -1 && dy == -1) return 8;
  return -1;
}

// Coarse parents of fine index x on a side of n cells: one (x even, or the
// last node of an odd side) or two neighbours at weight 1/2 (odd x < n).
struct Par1 {
  int a, b;  // a == b: single parent
};
__device__ inline Par1 parents1(int x, int n) {
  if (!(x & 1)) return Par1{x >> 1, x >> 1};
  if (x == n) return Par1{(n + 1) >> 1, (n + 1) >> 1};
  return Par1{(x - 1) >> 1, (x + 1) >> 1};
}
// fine index of coarse index I on a side of n fine cells
__device__ inline int fine_of(int I, int n) { return min(2 * I, n); }

// Bilinear interpolation of the coarse vector ec (row length cnx + 1) at fine
// node (x, y) of a level with fnx x fny cells.  (The level-1 operator couples
// the four vertices of a grid cell alike; interpolating along one diagonal
// only costs 3-5 CG iterations: P3 160^2 18 instead of 15.)
__device__ inline double prolong_at(int fnx, int fny, int cnx, const double* ec, int x, int y) {
  const Par1 px = parents1(x, fnx), py = parents1(y, fny);
  const int64_t cs = cnx + 1;
  const double lo = px.a == px.b ? ec[py.a * cs + px.a] : 0.5 * (ec[py.a * cs + px.a] + ec[py.a * cs + px.b]);
  if (py.a == py.b) return lo;
  const double hi = px.a == px.b ? ec[py.b * cs + px.a] : 0.5 * (ec[py.b * cs + px.a] + ec[py.b * cs + px.b]);
  return 0.5 * (lo + hi);
}

// weight of coarse node (I, J) in prolong_at at fine node (x, y)
__device__ inline double pweight(int fnx, int fny, int x, int y, int I, int J) {
  const Par1 px = parents1(x, fnx), py = parents1(y, fny);
  const double wx = px.a == px.b ? (px.a == I ? 1.0 : 0.0) : (px.a == I || px.b == I ? 0.5 : 0.0);
  const double wy = py.a == py.b ? (py.a == J ? 1.0 : 0.0) : (py.a == J || py.b == J ? 0.5 : 0.0);
  return wx * wy;
}

// ------------------------------------------------------------ set-up
// Galerkin coarse stencil R A P on the next level: R = P^T with the weights
// of prolong_at.  Eight lanes per coarse node: lane t takes the fine node at
// support offset t (lane 0 the ninth too), and a fixed shuffle tree sums the
// lanes' stencils.
template <class VS>
__global__ __launch_bounds__(256) void mg_rap_kernel(VS sel) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int64_t gid = (int64_t)lb * blockDim.x + threadIdx.x;
  const int64_t C = gid >> 3;
  const int t = (int)(gid & 7);
  const int cnx = Cc.nx, fnx = F.nx, fny = F.ny;
  const bool live = C < Cc.n;
  const int I = live ? (int)(C % (cnx + 1)) : 0, J = live ? (int)(C / (cnx + 1)) : 0;
  const unsigned char cm = live ? Cc.mask[C] : 1;  // written by mg_cmask_kernel
  double st[kStencil] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int o = t; !cm && o < kStencil; o += 8) {
    const int fx = fine_of(I, fnx) + kOffX[o], fy = fine_of(J, fny) + kOffY[o];
    const int64_t fi = (int64_t)fy * (fnx + 1) + fx;
    const bool in = fx >= 0 && fx <= fnx && fy >= 0 && fy <= fny && !F.mask[fi];
    const double w1 = in ? pweight(fnx, fny, fx, fy, I, J) : 0.0;
    if (w1 == 0.0) continue;
    for (int s = 0; s < kStencil; ++s) {
      const double av = F.a[s * F.n + fi];
      if (av == 0.0) continue;
      const int gx = fx + kOffX[s], gy = fy + kOffY[s];
      if (gx < 0 || gx > fnx || gy < 0 || gy > fny) continue;
      if (F.mask[(int64_t)gy * (fnx + 1) + gx]) continue;
      // coarse parents of fine node g, as prolong_at weighs them
      const Par1 px = parents1(gx, fnx), py = parents1(gy, fny);
      const int mx = px.a == px.b ? 1 : 2, my = py.a == py.b ? 1 : 2;
      const double w2 = (mx == 1 ? 1.0 : 0.5) * (my == 1 ? 1.0 : 0.5);
      for (int v = 0; v < my; ++v)
        for (int u = 0; u < mx; ++u) {
          const int qx = u ? px.b : px.a, qy = v ? py.b : py.a;
          if (Cc.mask[(int64_t)qy * (cnx + 1) + qx]) continue;  // zero column of P
          const int sl = slot_of(qx - I, qy - J);
#pragma unroll
          for (int k = 0; k < kStencil; ++k)
            if (k == sl) st[k] = fma(w1 * av, w2, st[k]);
        }
    }
  }
#pragma unroll
  for (int u = 0; u < kStencil; ++u) {
    st[u] += __shfl_xor(st[u], 1, 8);
    st[u] += __shfl_xor(st[u], 2, 8);
    st[u] += __shfl_xor(st[u], 4, 8);
  }
  if (t != 0 || !live) return;
#pragma unroll
  for (int u = 0; u < kStencil; ++u) Cc.a[u * Cc.n + C] = cm ? (u == 0 ? 1.0 : 0.0) : st[u];
  Cc.dinv[C] = cm ? 0.0 : 1.0 / st[0];
}

// Inverse of the coarsest operator (at most kCoarseDirect nodes), by
// Gauss-Jordan with partial pivoting on [A | I] in LDS: one thread per entry,
// the pivot row chosen by thread 0.  Fixed nodes have identity rows.
// Block b inverts the coarsest level of Ms[b] (skipped above kCoarseDirect).
__global__ __launch_bounds__(1024) void mg_coarse_inverse_kernel(const MgData* __restrict__ Ms) {
  constexpr int W = 2 * kCoarseDirect;
  __shared__ double m[kCoarseDirect * W];
  __shared__ int piv;
  const MgData& M = Ms[blockIdx.x];
  const MgLevel& L = M.lev[M.nlev - 1];
  double* const cinv = M.cinv;
  const int n = (int)L.n;
  if (n > kCoarseDirect) return;
  for (int e = threadIdx.x; e < n * W; e += blockDim.x) m[e] = 0.0;
  __syncthreads();
  for (int v = threadIdx.x; v < n; v += blockDim.x) {
    const int i = v % (L.nx + 1), j = v / (L.nx + 1);
    m[v * W + n + v] = 1.0;
    for (int s = 0; s < kStencil; ++s) {
      const int gx = i + kOffX[s], gy = j + kOffY[s];
      if (gx < 0 || gx > L.nx || gy < 0 || gy > L.ny) continue;
      m[v * W + gy * (L.nx + 1) + gx] += L.a[s * L.n + v];
    }
  }
  __syncthreads();
  for (int c = 0; c < n; ++c) {
    if (threadIdx.x == 0) {
      int best = c;
      for (int r = c + 1; r < n; ++r)
        if (fabs(m[r * W + c]) > fabs(m[best * W + c])) best = r;
      piv = best;
    }
    __syncthreads();
    const int pr = piv;
    if (pr != c)
      for (int e = threadIdx.x; e < 2 * n; e += blockDim.x) {
        const double a = m[c * W + e];
        m[c * W + e] = m[pr * W + e];
        m[pr * W + e] = a;
      }
    __syncthreads();
    const double pv = m[c * W + c];
    // each thread owns one (row, column) entry of the update
    double upd = 0.0;
    const int row = threadIdx.x / (2 * n), col = threadIdx.x % (2 * n);
    const bool own = threadIdx.x < n * 2 * n;
    if (own) {
      const double pc = m[c * W + col] / pv;
      upd = row == c ? pc : m[row * W + col] - m[row * W + c] * pc;
    }
    __syncthreads();
    if (own) m[row * W + col] = upd;
    __syncthreads();
  }
  for (int e = threadIdx.x; e < n * n; e += blockDim.x) cinv[e] = m[(e / n) * W + n + e % n];
}

// LDS image of the tail levels: per level its stencils (kStencil n) then
// dinv (n); blockIdx.y selects the hierarchy Ms[y].
__global__ void mg_tailpack_kernel(const MgData* __restrict__ Ms) {
  const MgData& M = Ms[blockIdx.y];
  int o = 0;
  for (int l = M.tail; l < M.nlev; ++l) {
    const int n = (int)M.lev[l].n;
    for (int u = blockIdx.x * blockDim.x + threadIdx.x; u < (kStencil + 1) * n; u += gridDim.x * blockDim.x)
      M.tailpack[o + u] = u < kStencil * n ? M.lev[l].a[u] : M.lev[l].dinv[u - kStencil * n];
    o += (kStencil + 1) * n;
  }
}

// Coarse masks (a coarse node is fixed when its fine node is), written
// before mg_rap_kernel reads the masks of neighbouring nodes.
template <class VS>
__global__ void mg_cmask_kernel(VS sel) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int64_t C = (int64_t)lb * blockDim.x + threadIdx.x;
  if (C >= Cc.n) return;
  const int I = (int)(C % (Cc.nx + 1)), J = (int)(C / (Cc.nx + 1));
  Cc.mask[C] = F.mask[(int64_t)fine_of(J, F.ny) * (F.nx + 1) + fine_of(I, F.nx)];
}

// ------------------------------------------------------- vertex levels
// (A x)_v on a level, with x given as a function of (index, i, j), so that
// fused kernels can form x on the fly.
template <class X>
__device__ inline double stencil_apply(const MgLevel& L, int64_t v, int i, int j, const X& xv) {
  const int64_t row = L.nx + 1;
  double s = L.a[v] * xv(v, i, j);
  if (i < L.nx) s = fma(L.a[L.n + v], xv(v + 1, i + 1, j), s);
  if (i > 0) s = fma(L.a[2 * L.n + v], xv(v - 1, i - 1, j), s);
  if (j < L.ny) s = fma(L.a[3 * L.n + v], xv(v + row, i, j + 1), s);
  if (j > 0) s = fma(L.a[4 * L.n + v], xv(v - row, i, j - 1), s);
  if (i < L.nx && j > 0) s = fma(L.a[5 * L.n + v], xv(v + 1 - row, i + 1, j - 1), s);
  if (i > 0 && j < L.ny) s = fma(L.a[6 * L.n + v], xv(v - 1 + row, i - 1, j + 1), s);
  if (i < L.nx && j < L.ny) s = fma(L.a[7 * L.n + v], xv(v + 1 + row, i + 1, j + 1), s);
  if (i > 0 && j > 0) s = fma(L.a[8 * L.n + v], xv(v - 1 - row, i - 1, j - 1), s);
  return s;
}

// The vertex-level kernels take a selector (VOne, VGroup) that names the
// instance of the block: its fine level F, coarse level C and CG state.

// two pre-smoothing sweeps from zero in one pass: e1 = om dinv r is formed at
// the neighbours on the fly, e = e1 + om dinv (r - A e1)
template <class VS>
__global__ __launch_bounds__(256) void v_pre_kernel(VS sel, double om) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  if (R.st->done) return;
  const MgLevel& L = R.F;
  const int64_t v = (int64_t)lb * blockDim.x + threadIdx.x;
  if (v >= L.n) return;
  const int i = (int)(v % (L.nx + 1)), j = (int)(v / (L.nx + 1));
  auto e1 = [&](int64_t u, int, int) { return om * L.dinv[u] * L.r[u]; };
  L.e[v] = e1(v, i, j) + om * L.dinv[v] * (L.r[v] - stencil_apply(L, v, i, j, e1));
}

// second post-smoothing sweep: e = t + om dinv (r - A t)
template <class VS>
__global__ __launch_bounds__(256) void v_smooth_kernel(VS sel, double om) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  if (R.st->done) return;
  const MgLevel& L = R.F;
  const int64_t v = (int64_t)lb * blockDim.x + threadIdx.x;
  if (v >= L.n) return;
  const int i = (int)(v % (L.nx + 1)), j = (int)(v / (L.nx + 1));
  const double* __restrict__ in = L.t;
  auto xv = [&](int64_t u, int, int) { return in[u]; };
  L.e[v] = in[v] + om * L.dinv[v] * (L.r[v] - stencil_apply(L, v, i, j, xv));
}

// fine residual r - A e at (fx, fy); 0 outside the grid and on fixed nodes.
// With one_sweep the smoothed iterate is the single sweep from zero,
// e = om dinv r, formed on the fly.
__device__ inline double fine_res(const MgLevel& F, int fx, int fy, bool one_sweep, double om) {
  if (fx < 0 || fx > F.nx || fy < 0 || fy > F.ny) return 0.0;
  const int64_t fi = (int64_t)fy * (F.nx + 1) + fx;
  if (F.mask[fi]) return 0.0;
  if (one_sweep) {
    auto e1 = [&](int64_t u, int, int) { return om * F.dinv[u] * F.r[u]; };
    return F.r[fi] - stencil_apply(F, fi, fx, fy, e1);
  }
  auto ev = [&](int64_t u, int, int) { return F.e[u]; };
  return F.r[fi] - stencil_apply(F, fi, fx, fy, ev);
}

// coarse r = R (r - A e), R = P^T: the fine node of C and its eight stencil
// neighbours, weighted as prolong_at weighs C there.  Eight lanes per
// coarse node: lane t forms the fine residual at stencil offset t (lane 0
// the ninth too), and a fixed shuffle tree sums them.
template <class VS>
__global__ __launch_bounds__(256) void v_restrict_kernel(VS sel, int one_sweep, double om) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  if (R.st->done) return;
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int64_t g = (int64_t)lb * blockDim.x + threadIdx.x;
  const int64_t C = g >> 3;
  const int t = (int)(g & 7);
  double val = 0.0;
  if (C < Cc.n && !Cc.mask[C]) {
    const int I = (int)(C % (Cc.nx + 1)), J = (int)(C / (Cc.nx + 1));
    for (int o = t; o < kStencil; o += 8) {
      const int x = fine_of(I, F.nx) + kOffX[o], y = fine_of(J, F.ny) + kOffY[o];
      const double w = (x < 0 || x > F.nx || y < 0 || y > F.ny) ? 0.0 : pweight(F.nx, F.ny, x, y, I, J);
      if (w != 0.0) val = fma(w, fine_res(F, x, y, one_sweep != 0, om), val);
    }
  }
  val += __shfl_xor(val, 1, 8);
  val += __shfl_xor(val, 2, 8);
  val += __shfl_xor(val, 4, 8);
  if (t == 0 && C < Cc.n) Cc.r[C] = val;
}

// prolongation and the first post-smoothing sweep in one pass:
// e' = e + P ec on free nodes (formed at the neighbours on the fly),
// out = e' + om dinv (r - A e').  With one_sweep the pre-smoothed iterate is
// e = om dinv r (formed on the fly) and out is the level's final e.
template <class VS>
__global__ __launch_bounds__(256) void v_post_kernel(VS sel, int one_sweep, double om) {
  int lb;
  const VRec& R = vrec_of(sel, lb);
  if (R.st->done) return;
  const MgLevel& F = R.F;
  const MgLevel& Cc = R.C;
  const int64_t v = (int64_t)lb * blockDim.x + threadIdx.x;
  if (v >= F.n) return;
  const int i = (int)(v % (F.nx + 1)), j = (int)(v / (F.nx + 1));
  if (one_sweep) {
    auto ep = [&](int64_t u, int x, int y) {
      const double e = om * F.dinv[u] * F.r[u];
      return F.mask[u] ? e : e + prolong_at(F.nx, F.ny, Cc.nx, Cc.e, x, y);
    };
    F.e[v] = ep(v, i, j) + om * F.dinv[v] * (F.r[v] - stencil_apply(F, v, i, j, ep));
  } else {
    auto ep = [&](int64_t u, int x, int y) {
      return F.mask[u] ? F.e[u] : F.e[u] + prolong_at(F.nx, F.ny, Cc.nx, Cc.e, x, y);
    };
    F.t[v] = ep(v, i, j) + om * F.dinv[v] * (F.r[v] - stencil_apply(F, v, i, j, ep));
  }
}

// Coarsest level too large for v_tail_kernel: `sweeps` damped Jacobi sweeps
// from zero in one block, vectors in global memory.
__global__ __launch_bounds__(1024) void v_coarsest_kernel(MgLevel L, double om, int sweeps, const CgState* st) {
  if (st->done) return;
  for (int64_t v = threadIdx.x; v < L.n; v += blockDim.x) L.e[v] = om * L.dinv[v] * L.r[v];
  __syncthreads();
  for (int it = 1; it < sweeps; ++it) {
    for (int64_t v = threadIdx.x; v < L.n; v += blockDim.x) {
      const int i = (int)(v % (L.nx + 1)), j = (int)(v / (L.nx + 1));
      auto xv = [&](int64_t u, int, int) { return L.e[u]; };
      L.t[v] = L.e[v] + om * L.dinv[v] * (L.r[v] - stencil_apply(L, v, i, j, xv));
    }
    __syncthreads();
    for (int64_t v = threadIdx.x; v < L.n; v += blockDim.x) L.e[v] = L.t[v];
    __syncthreads();
  }
}

// Level of the one-workgroup tail: stencils, diagonal inverse and vectors
// all in LDS.  A fixed node has dinv = 0 (its stencil row is the identity).
struct TailLevel {
  int nx, ny, n;
  const double* a;     // a[s*n + v]
  const double* dinv;
};

__device__ inline double tail_apply(const TailLevel& L, const double* x, int v, int i, int j) {
  const int row = L.nx + 1;
  double s = L.a[v] * x[v];
  if (i < L.nx) s = fma(L.a[L.n + v], x[v + 1], s);
  if (i > 0) s = fma(L.a[2 * L.n + v], x[v - 1], s);
  if (j < L.ny) s = fma(L.a[3 * L.n + v], x[v + row], s);
  if (j > 0) s = fma(L.a[4 * L.n + v], x[v - row], s);
  if (i < L.nx && j > 0) s = fma(L.a[5 * L.n + v], x[v + 1 - row], s);
  if (i > 0 && j < L.ny) s = fma(L.a[6 * L.n + v], x[v - 1 + row], s);
  if (i < L.nx && j < L.ny) s = fma(L.a[7 * L.n + v], x[v + 1 + row], s);
  if (i > 0 && j > 0) s = fma(L.a[8 * L.n + v], x[v - 1 - row], s);
  return s;
}

// one Jacobi sweep: out = in + om dinv (r - A in)
__device__ inline void tail_sweep(const TailLevel& L, const double* in, double* out, const double* r, double om) {
  for (int v = threadIdx.x; v < L.n; v += blockDim.x) {
    const int i = v % (L.nx + 1), j = v / (L.nx + 1);
    out[v] = in[v] + om * L.dinv[v] * (r[v] - tail_apply(L, in, v, i, j));
  }
}

// Levels lt = tail .. nlev-1 of the V-cycle in one workgroup (their sizes
// sum to at most kTailNodes), everything in LDS: reads lev[lt].r, writes
// lev[lt].e.  Block b serves the hierarchy Ms[b] with CG state sts[b] (one
// block for a single problem, one per instance for a group).
// Same sweeps as the per-level kernels: two pre-smoothing sweeps,
// restriction of the residual, coarse_sweeps sweeps on the coarsest level,
// prolongation and two post-smoothing sweeps.
__global__ __launch_bounds__(kTailThreads) void v_tail_kernel(const MgData* __restrict__ Ms, const CgState* sts) {
  __shared__ double pool[(kStencil + 4) * kTailNodes];
  const MgData& M = Ms[blockIdx.x];
  if (sts[blockIdx.x].done) return;
  const int lt = M.tail;
  const double om = M.omega_v;
  double* const E = pool;                    // scratch / residual
  double* const Tt = pool + kTailNodes;      // iterate
  double* const R = pool + 2 * kTailNodes;   // right-hand sides
  double* const SA = pool + 3 * kTailNodes;  // stencils (kStencil n) and dinv (n) per level
  {
    int tn = 0;
    for (int l = lt; l < M.nlev; ++l) tn += (int)M.lev[l].n;
    const double* __restrict__ src = M.tailpack;
#pragma unroll 8
    for (int u = threadIdx.x; u < (kStencil + 1) * tn; u += blockDim.x) SA[u] = src[u];
  }
  {
    const MgLevel L = M.lev[lt];
    for (int v = threadIdx.x; v < (int)L.n; v += blockDim.x) R[v] = L.r[v];
  }
  __syncthreads();
  // level l's stencil block starts at (kStencil + 1) * (nodes of levels lt..l-1); its
  // vectors at the same node offset o
  auto lvl = [&](int l, int o) {
    TailLevel L;
    L.nx = M.lev[l].nx;
    L.ny = M.lev[l].ny;
    L.n = (int)M.lev[l].n;
    L.a = SA + (kStencil + 1) * o;
    L.dinv = SA + (kStencil + 1) * o + kStencil * L.n;
    return L;
  };
  int o = 0;
  for (int l = lt; l < M.nlev - 1; ++l) {
    const TailLevel L = lvl(l, o);
    const TailLevel Cc = lvl(l + 1, o + L.n);
    double *e = E + o, *t = Tt + o, *r = R + o;
    if (M.vsweeps > 1) {
      for (int v = threadIdx.x; v < L.n; v += blockDim.x) e[v] = om * L.dinv[v] * r[v];
      __syncthreads();
      tail_sweep(L, e, t, r, om);
    } else {
      for (int v = threadIdx.x; v < L.n; v += blockDim.x) t[v] = om * L.dinv[v] * r[v];
    }
    __syncthreads();
    for (int v = threadIdx.x; v < L.n; v += blockDim.x) {
      const int i = v % (L.nx + 1), j = v / (L.nx + 1);
      e[v] = L.dinv[v] == 0.0 ? 0.0 : r[v] - tail_apply(L, t, v, i, j);
    }
    __syncthreads();
    double* rc = R + o + L.n;
    for (int C = threadIdx.x; C < Cc.n; C += blockDim.x) {
      double s = 0.0;
      if (Cc.dinv[C] != 0.0) {
        const int I = C % (Cc.nx + 1), J = C / (Cc.nx + 1);
        const int x = fine_of(I, L.nx), y = fine_of(J, L.ny);
        auto res = [&](int fx, int fy) {
          return (fx < 0 || fx > L.nx || fy < 0 || fy > L.ny)
                     ? 0.0
                     : pweight(L.nx, L.ny, fx, fy, I, J) * e[fy * (L.nx + 1) + fx];
        };
        s = res(x, y) + res(x + 1, y) + res(x - 1, y) + res(x, y + 1) + res(x, y - 1) + res(x + 1, y - 1) +
            res(x - 1, y + 1) + res(x + 1, y + 1) + res(x - 1, y - 1);
      }
      rc[C] = s;
    }
    __syncthreads();
    o += L.n;
  }
  // coarsest level
  double* ec;
  {
    const TailLevel L = lvl(M.nlev - 1, o);
    double *e = E + o, *t = Tt + o;
    const double* r = R + o;
    if (L.n <= kCoarseDirect) {
      // exact solve with the inverse computed at set-up
      for (int v = threadIdx.x; v < L.n; v += blockDim.x) {
        double acc = 0.0;
        for (int u = 0; u < L.n; ++u) acc = fma(M.cinv[v * L.n + u], r[u], acc);
        t[v] = acc;
      }
      __syncthreads();
    } else {
      for (int v = threadIdx.x; v < L.n; v += blockDim.x) t[v] = om * L.dinv[v] * r[v];
      __syncthreads();
      for (int it = 1; it < M.coarse_sweeps; ++it) {
        tail_sweep(L, t, e, r, om);
        __syncthreads();
        double* sw = e;
        e = t;
        t = sw;
      }
    }
    ec = t;
  }
  for (int l = M.nlev - 2; l >= lt; --l) {
    const int oc = o;
    o -= (int)M.lev[l].n;
    const TailLevel L = lvl(l, o);
    const TailLevel Cc = lvl(l + 1, oc);
    double *e = E + o, *t = Tt + o;
    const double* r = R + o;
    for (int v = threadIdx.x; v < L.n; v += blockDim.x) {
      if (L.dinv[v] == 0.0) continue;
      t[v] += prolong_at(L.nx, L.ny, Cc.nx, ec, v % (L.nx + 1), v / (L.nx + 1));
    }
    __syncthreads();
    if (M.vsweeps > 1) {
      tail_sweep(L, t, e, r, om);
      __syncthreads();
      tail_sweep(L, e, t, r, om);
      __syncthreads();
      ec = t;
    } else {
      tail_sweep(L, t, e, r, om);
      __syncthreads();
      ec = e;
    }
  }
  {
    const MgLevel L = M.lev[lt];
    for (int v = threadIdx.x; v < (int)L.n; v += blockDim.x) L.e[v] = ec[v];
  }
}

int grid1(int64_t n, int t = 256) {
  int64_t g = (n + t - 1) / t;
  if (g < 1) g = 1;
  if (g > (1 << 30)) g = 1 << 30;
  return (int)g;
}

// V-cycle from level l down; the result is left in lev[l].e.  dM is the
// device copy of M that the tail kernel reads.
int vcycle(const MgData& M, const MgData* dM, int l, const CgState* st, hipStream_t s) {
  if (l >= M.tail) {
    hipLaunchKernelGGL(v_tail_kernel, dim3(1), dim3(kTailThreads), 0, s, dM, st);
    return (int)hipGetLastError();
  }
  const MgLevel& L = M.lev[l];
  const double om = M.omega_v;
  if (l == M.nlev - 1) {
    hipLaunchKernelGGL(v_coarsest_kernel, dim3(1), dim3(1024), 0, s, L, om, M.coarse_sweeps, st);
    return (int)hipGetLastError();
  }
  const MgLevel& Cc = M.lev[l + 1];
  const VOne one_rec{VRec{L, Cc, st}};
  const int g = grid1(L.n);
  const int one = M.vsweeps > 1 ? 0 : 1;
  if (!one) hipLaunchKernelGGL(v_pre_kernel<VOne>, dim3(g), dim3(256), 0, s, one_rec, om);
  hipLaunchKernelGGL(v_restrict_kernel<VOne>, dim3(grid1(8 * Cc.n)), dim3(256), 0, s, one_rec, one, om);
  int e = vcycle(M, dM, l + 1, st, s);
  if (e) return e;
  hipLaunchKernelGGL(v_post_kernel<VOne>, dim3(g), dim3(256), 0, s, one_rec, one, om);
  if (!one) hipLaunchKernelGGL(v_smooth_kernel<VOne>, dim3(g), dim3(256), 0, s, one_rec, om);
  return (int)hipGetLastError();
}

// The same V-cycle for every instance of a group: depth by depth down to the
// tails, every tail in one launch (one workgroup each), depth by depth up.
// An instance whose tail starts at depth t takes part in depths 1..t-1 only.
int vcycle_group(const MgGroup& G, hipStream_t s) {
  const int one = G.vsweeps > 1 ? 0 : 1;
  const double om = G.omega_v;
  for (int d = 1; d < G.ndepth; ++d) {
    if (!one) hipLaunchKernelGGL(v_pre_kernel<VGroup>, dim3(G.gnode[d]), dim3(256), 0, s, G.node[d], om);
    hipLaunchKernelGGL(v_restrict_kernel<VGroup>, dim3(G.gres[d]), dim3(256), 0, s, G.res[d], one, om);
  }
  hipLaunchKernelGGL(v_tail_kernel, dim3(G.ninst), dim3(kTailThreads), 0, s, G.dM, (const CgState*)G.st);
  for (int d = G.ndepth - 1; d >= 1; --d) {
    hipLaunchKernelGGL(v_post_kernel<VGroup>, dim3(G.gnode[d]), dim3(256), 0, s, G.node[d], one, om);
    if (!one) hipLaunchKernelGGL(v_smooth_kernel<VGroup>, dim3(G.gnode[d]), dim3(256), 0, s, G.node[d], om);
  }
  return (int)hipGetLastError();
}

}  // namespace

int mg_setup_levels(const MgData& M, const MgData* dM, hipStream_t s) {
  for (int l = 1; l + 1 < M.nlev; ++l) {
    const VOne rec{VRec{M.lev[l], M.lev[l + 1], nullptr}};
    hipLaunchKernelGGL(mg_cmask_kernel<VOne>, dim3(grid1(M.lev[l + 1].n)), dim3(256), 0, s, rec);
    hipLaunchKernelGGL(mg_rap_kernel<VOne>, dim3(grid1(8 * M.lev[l + 1].n)), dim3(256), 0, s, rec);
  }
  hipLaunchKernelGGL(mg_coarse_inverse_kernel, dim3(1), dim3(1024), 0, s, dM);
  if (M.tail < M.nlev) hipLaunchKernelGGL(mg_tailpack_kernel, dim3(16, 1), dim3(256), 0, s, dM);
  return (int)hipGetLastError();
}

int mg_setup_levels_group(const MgSetupGroup& S, hipStream_t s) {
  for (int d = 1; d < S.ndepth; ++d) {
    hipLaunchKernelGGL(mg_cmask_kernel<VGroup>, dim3(S.gcmask[d]), dim3(256), 0, s, S.cmask[d]);
    hipLaunchKernelGGL(mg_rap_kernel<VGroup>, dim3(S.grap[d]), dim3(256), 0, s, S.rap[d]);
  }
  hipLaunchKernelGGL(mg_coarse_inverse_kernel, dim3(S.ninst), dim3(1024), 0, s, S.dM);
  hipLaunchKernelGGL(mg_tailpack_kernel, dim3(16, S.ninst), dim3(256), 0, s, S.dM);
  return (int)hipGetLastError();
}

int launch_vcycle(const MgData& M, const MgData* dM, const CgState* st, hipStream_t s) {
  return vcycle(M, dM, 1, st, s);
}
int launch_vcycle_group(const MgGroup& G, hipStream_t s) { return vcycle_group(G, s); }

}  // namespace hdg
