// The multigrid preconditioner on meshes without rectangle structure
// (hdg_amg.h).  Indexed gathers throughout; on the sizes it is used for the
// arrays stay in the caches and every kernel is bound by its launch and two
// or three dependent loads, so the cycle is built for few launches: seven per
// CG iteration while the levels below the vertices fit one workgroup.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <utility>

#include "hdg_amg.h"

namespace hdg {

namespace {

constexpr double kQ = 0.28867513459481288225;  // 1 / (2 sqrt 3)

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// ------------------------------------------------------------------ set-up
__global__ __launch_bounds__(256) void amg_fix_kernel(AmgTop A, TraceSystem T) {
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v >= A.n) return;
  bool fix = A.vp[v] == A.vp[v + 1];  // a node of no cell
  for (int e = A.vp[v]; e < A.vp[v + 1]; ++e) {
    const int code = A.vi[e];
    if ((code & 3) < 2)
      for (int i = 0; i < T.nt; ++i) fix |= T.dmask[(int64_t)(code >> 2) * T.nt + i] != 0;
  }
  A.vfix[v] = fix;
}

// Local index of vertex v in cell c (-1: not there), and the weight of mode 1
// of v's hat function on the cell's face lf (v an end of it; the face runs from
// its lower node id to the higher in either cell).
__device__ __forceinline__ int local_of(const int* __restrict__ cv, int64_t c, int v) {
  return cv[3 * c] == v ? 0 : (cv[3 * c + 1] == v ? 1 : (cv[3 * c + 2] == v ? 2 : -1));
}
__device__ __forceinline__ double mode1(const int* __restrict__ cn, int64_t c, int lv, int lf) {
  return cn[3 * c + lv] > cn[3 * c + 3 - lv - lf] ? kQ : -kQ;
}

// (hat v)^T (-Ate_c) (hat w)
__device__ double cell_stiffness(const int* __restrict__ cn, const int* __restrict__ cv,
                                 const double* __restrict__ Ate, int nt, int64_t c, int v, int w) {
  const int lv = local_of(cv, c, v), lw = local_of(cv, c, w), ntr = 3 * nt;
  if (lv < 0 || lw < 0) return 0.0;
  const double* K = Ate + c * ntr * ntr;
  double s = 0.0;
#pragma unroll
  for (int a = 1; a < 3; ++a)
#pragma unroll
    for (int b = 1; b < 3; ++b) {
      const int lf = (lv + a) % 3, lg = (lw + b) % 3;
      const double p = mode1(cn, c, lv, lf), q = mode1(cn, c, lw, lg);
      const double* k = K + (lf * nt) * ntr + lg * nt;
      s += 0.5 * (0.5 * k[0] + q * k[1]) + p * (0.5 * k[ntr] + q * k[ntr + 1]);
    }
  return -s;
}

// Level 0's operator P^T S P, cell by cell: eight lanes per row.
__global__ __launch_bounds__(256) void amg_vertex_kernel(DevMesh m, int nt, const double* __restrict__ Ate, AmgTop A,
                                                         AmgLevel L) {
  const int v = (blockIdx.x * 256 + threadIdx.x) >> 3;
  if (v >= L.n) return;
  for (int e = L.ap[v] + (threadIdx.x & 7); e < L.ap[v + 1]; e += 8) {
    const int w = L.ai[e];
    double s = 0.0;
    if (!A.vfix[v] && !A.vfix[w]) {
      if (w != v) {
        const int64_t f = A.af[e];
        for (int k = 0; k < 2; ++k)
          if (m.fcell[2 * f + k] >= 0) s += cell_stiffness(m.cn, A.cv, Ate, nt, m.fcell[2 * f + k], v, w);
      } else {
        for (int u = A.vp[v]; u < A.vp[v + 1]; ++u) {  // the cells around v, by the faces opposite to it
          const int code = A.vi[u];
          if ((code & 3) >= 2)
            s += cell_stiffness(m.cn, A.cv, Ate, nt, m.fcell[2 * (code >> 2) + (code & 3) - 2], v, v);
        }
      }
    }
    L.av[e] = s;
  }
}

// G = P - w J S P: thread per trace row, vertex after vertex.
template <int NT>
__global__ __launch_bounds__(64 * NT) void amg_g_kernel(DevMesh m, TraceSystem T, const double* __restrict__ Ate,
                                                        AmgTop A) {
  constexpr int NTR = 3 * NT;
  __shared__ double rs[64 * NT];
  const int64_t r = (int64_t)blockIdx.x * (64 * NT) + threadIdx.x;
  const bool in = r < T.N;
  const int64_t f = in ? r / NT : 0;
  const int a = (int)(r - f * NT);
#pragma unroll 1
  for (int j = 0; j < 4; ++j) {
    const int v = A.fv[4 * f + j];
    const bool on = in && v >= 0 && !A.vfix[v];
    double s = 0.0;
    if (on) {
      for (int k = 0; k < 2; ++k) {
        const int64_t c = m.fcell[2 * f + k];
        if (c < 0) continue;
        const int lv = local_of(A.cv, c, v);
        const int l = m.cf[3 * c] == f ? 0 : (m.cf[3 * c + 1] == f ? 1 : (m.cf[3 * c + 2] == f ? 2 : -1));
        if (lv < 0 || l < 0) continue;
        const double* K = Ate + c * (NTR * NTR) + (l * NT + a) * NTR;
#pragma unroll
        for (int b = 1; b < 3; ++b) {
          const int lg = (lv + b) % 3;
          s -= 0.5 * K[lg * NT] + mode1(m.cn, c, lv, lg) * K[lg * NT + 1];
        }
      }
    }
    double p = 0.0;
    if (on && j < 2) p = a == 0 ? 0.5 : (a == 1 ? (j ? kQ : -kQ) : 0.0);
    jacobi_apply<NT>(T.Dinv, T.nf, rs, s, r, in,
                     [&](double y) { A.g[(int64_t)j * T.N + r] = on ? fma(-kAmgOmega, y, p) : 0.0; });
  }
}

// Position of column c in a sorted row, or -1.
__device__ __forceinline__ int find(const int* __restrict__ idx, int lo, int hi, int c) {
  for (int e = lo; e < hi; ++e)
    if (idx[e] == c) return e;
  return -1;
}

// Sum over the eight lanes of a row.
__device__ __forceinline__ double sum8(double s) {
  s += __shfl_xor(s, 1, 8);
  s += __shfl_xor(s, 2, 8);
  s += __shfl_xor(s, 4, 8);
  return s;
}

// D of a level, and (transfer) its smoothed interpolation P = (I - w D A) P0,
// P0 the aggregates' indicator on the free rows, on G's pattern: eight lanes
// per row (the set-up kernels with a thread per row took 32, 133 and, the
// product below at 16 lanes, 152 us at 7872 and 770 nodes).
__global__ __launch_bounds__(256) void amg_p_kernel(AmgLevel L, int transfer) {
  const int u = (blockIdx.x * 256 + threadIdx.x) >> 3, t = threadIdx.x & 7;
  const bool on = u < L.n;
  const int v = on ? u : 0, e0 = L.ap[v], e1 = L.ap[v + 1];
  double d = 0.0, s = 0.0;
  for (int e = e0 + t; e < e1; e += 8) {
    const double a = L.av[e];
    s += fabs(a);
    if (L.ai[e] == v) d = a;
  }
  d = sum8(d);
  s = sum8(s);
  const double D = d > 0.0 ? 1.0 / fmax(d, 0.5 * s) : 0.0;
  if (!on) return;
  if (t == 0) L.dinv[v] = kAmgOmegaV * D;
  if (!transfer) return;
  for (int q = L.gp[v] + t; q < L.gp[v + 1]; q += 8) {
    const int c = L.gi[q];
    double x = 0.0;
    for (int e = e0; e < e1; ++e)
      if (L.agg[L.ai[e]] == c) x += L.av[e];
    L.pv[q] = D == 0.0 ? 0.0 : fma(-kAmgOmegaP * D, x, L.agg[v] == c ? 1.0 : 0.0);
  }
}

// A P and G = P - w D A P: eight lanes per row, an entry each.
__global__ __launch_bounds__(256) void amg_ap_kernel(AmgLevel L) {
  const int v = (blockIdx.x * 256 + threadIdx.x) >> 3;
  if (v >= L.n) return;
  const double wd = L.dinv[v];
  for (int q = L.gp[v] + (threadIdx.x & 7); q < L.gp[v + 1]; q += 8) {
    const int c = L.gi[q];
    double t = 0.0;
    for (int e = L.ap[v]; e < L.ap[v + 1]; ++e) {
      const int w = L.ai[e], x = find(L.gi, L.gp[w], L.gp[w + 1], c);
      if (x >= 0) t = fma(L.av[e], L.pv[x], t);
    }
    L.apv[q] = t;
    L.gv[q] = fma(-wd, t, L.pv[q]);
  }
}

// The next level's operator P^T (A P): a workgroup per row, 16 entries at a
// time, the sum over the fine rows split 16 ways and added up in LDS.
__global__ __launch_bounds__(256) void amg_rap_kernel(AmgLevel L, AmgLevel C) {
  __shared__ double sh[256];
  const int c = blockIdx.x, part = threadIdx.x >> 4;
  for (int e0 = C.ap[c]; e0 < C.ap[c + 1]; e0 += 16) {
    const int e = e0 + (threadIdx.x & 15);
    double s = 0.0;
    if (e < C.ap[c + 1]) {
      const int d = C.ai[e];
      for (int t = L.tp[c] + part; t < L.tp[c + 1]; t += 16) {
        const int v = L.ti[t];
        const double p = L.pv[L.tx[t]];
        if (p == 0.0) continue;
        const int x = find(L.gi, L.gp[v], L.gp[v + 1], d);
        if (x >= 0) s = fma(p, L.apv[x], s);
      }
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < 16 && e < C.ap[c + 1]) {
      for (int k = 1; k < 16; ++k) s += sh[threadIdx.x + 16 * k];
      C.av[e] = s;
    }
    __syncthreads();
  }
}

// Inverse of the last operator (n <= kAmgDirect; SPD on the rows with a
// positive diagonal, identity rows elsewhere; singular without any fixed
// vertex, see kNoPivot): Gauss-Jordan without pivoting,
// 6 x 6 entries per thread in registers, the pivot's row and column updated by
// the same fma as the rest (factors p - 1 and 1 + 1/p, p the pivot).
__global__ __launch_bounds__(256) void amg_inverse_kernel(AmgLevel L, double* __restrict__ cinv) {
  constexpr int T = 16, E = kAmgDirect / T;
  __shared__ double full[kAmgDirect * kAmgDirect];
  __shared__ double rowb[2][kAmgDirect], colb[2][kAmgDirect], mean[kAmgDirect + 1];
  __shared__ int fixed, dropped;
  const int n = L.n, tr = threadIdx.x / T, tc = threadIdx.x % T;
  if (threadIdx.x == 0) fixed = dropped = 0;
  for (int i = threadIdx.x; i < n * n; i += 256) full[i] = 0.0;
  __syncthreads();
  for (int v = threadIdx.x; v < n; v += 256)
    for (int e = L.ap[v]; e < L.ap[v + 1]; ++e) full[v * n + L.ai[e]] += L.av[e];  // a vertex pair may have two entries
  __syncthreads();
  for (int v = threadIdx.x; v < n; v += 256) {
    if (!(full[v * n + v] > 0.0)) {
      full[v * n + v] = 1.0;
      fixed = 1;
    }
  }
  __syncthreads();
  double m[E][E], least[E];  // the entries, and the least pivots of those on the diagonal
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int b = 0; b < E; ++b) {
      const int r = tr + T * a, c = tc + T * b;
      m[a][b] = r < n && c < n ? full[r * n + c] : 0.0;
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
      if (r < n && c < n) cinv[r * n + c] = m[a][b];
    }
  if (dropped && !fixed) project_constants(cinv, n, mean);
}

// ------------------------------------------------------------------- cycle
// The first kernel of a cycle, two parts side by side: blocks [0, nbv)
// restrict, r_0 = G^T r at eight lanes per vertex (a face's NT values lie
// together in G as in r); the others form t = 2 w z - w^2 J S z, z = J r.
// Takes the next product's convergence test (maxit >= 0), so that a converged
// solve skips its last cycle, and reports a cycle that was not definite ((r,
// z) <= 0) as a breakdown; the lead block records the state.
template <int NT>
__global__ __launch_bounds__(64 * NT) void amg_first_kernel(DevPattern P, TraceSystem T, CgVectors v, AmgTop A,
                                                            int nbv, double rtol2, int maxit) {
  constexpr int NTH = 64 * NT;
  __shared__ double rs[NTH];
  __shared__ double sh[NT];
  CgState* st = v.st;
  if (st->done) return;
  double part = 0.0;
  if (maxit >= 0)
    for (int i = threadIdx.x; i < v.nblocks; i += NTH) part += v.part[(size_t)3 * v.nblocks + i];
  part = wave_sum(part);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = part;
  __syncthreads();
  if (maxit >= 0) {
    double rr = 0.0;
#pragma unroll
    for (int w = 0; w < NT; ++w) rr += sh[w];
    const int it = st->i_spmv - 1;
    const bool conv = rr <= rtol2 * st->bb, indefinite = !(st->rz[it & 1] > 0.0);
    if (conv || indefinite || it >= maxit) {
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->it = it;
        st->rr = rr;
        st->done = conv ? 1 : (indefinite ? 3 : 2);
      }
      return;
    }
  }
  if ((int)blockIdx.x < nbv) {
    const int u = blockIdx.x * (NTH / 8) + (threadIdx.x >> 3);
    const bool on = u < A.n;
    double s = 0.0;
    if (on) {
      for (int e = A.vp[u] + (threadIdx.x & 7); e < A.vp[u + 1]; e += 8) {
        const int code = A.vi[e];
        const int64_t f = (int64_t)(code >> 2) * NT;
        const double* g = A.g + (int64_t)(code & 3) * T.N + f;
        const double* r = v.r + f;
#pragma unroll
        for (int i = 0; i < NT; ++i) s = fma(g[i], r[i], s);
      }
    }
    s = sum8(s);
    if (on && (threadIdx.x & 7) == 0) A.r[u] = s;
    return;
  }
  const int64_t r = (int64_t)(blockIdx.x - nbv) * NTH + threadIdx.x;
  const bool in = r < T.N;
  double q = 0.0;
  const double* __restrict__ z = v.z;
  if (in) {
    const int64_t f = r / NT;
    double acc = 0.0;
    if constexpr (kSymBlocks<NT>) {
      acc = sym_row<NT>(P.nbr, T.blk, T.nf, f, (int)(r - f * NT), [&](int64_t g, int b) { return z[g * NT + b]; });
    } else {
      const int* bc = P.bcol + f * kSlots;
#pragma unroll
      for (int s = 0; s < kSlots; ++s) {
        const int64_t g = (int64_t)__ldg(bc + s) * NT;
#pragma unroll
        for (int b = 0; b < NT; ++b) acc = fma(T.vals[(int64_t)(s * NT + b) * T.N + r], z[g + b], acc);
      }
    }
    q = T.dmask[r] ? 0.0 : -acc;
  }
  jacobi_apply<NT>(T.Dinv, T.nf, rs, q, r, in,
                   [&](double y) { A.t[r] = fma(-kAmgOmega * kAmgOmega, y, 2.0 * kAmgOmega * z[r]); });
}

// Next level's r = G^T r: 16 lanes per row.
__global__ __launch_bounds__(256) void amg_restrict_kernel(AmgLevel L, AmgLevel C, const CgState* st) {
  if (st->done) return;
  const int c = (blockIdx.x * 256 + threadIdx.x) >> 4;
  const bool on = c < C.n;
  double s = 0.0;
  if (on)
    for (int t = L.tp[c] + (threadIdx.x & 15); t < L.tp[c + 1]; t += 16) s = fma(L.gv[L.tx[t]], L.r[L.ti[t]], s);
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 16);
  if (on && (threadIdx.x & 15) == 0) C.r[c] = s;
}

// e = 2 w D r - w D A w D r + G e_next: eight lanes per row (a thread per
// row: 7.1 us at 7872 nodes).
__global__ __launch_bounds__(256) void amg_post_kernel(AmgLevel L, const double* __restrict__ ec, const CgState* st) {
  if (st->done) return;
  const int u = (blockIdx.x * 256 + threadIdx.x) >> 3, t = threadIdx.x & 7;
  const bool on = u < L.n;
  const int v = on ? u : 0;
  const double wd = L.dinv[v];
  double s = 0.0, g = 0.0;
  for (int e = L.ap[v] + t; e < L.ap[v + 1]; e += 8) {
    const int w = L.ai[e];
    s = fma(L.av[e], L.dinv[w] * L.r[w], s);
  }
  for (int q = L.gp[v] + t; q < L.gp[v + 1]; q += 8) g = fma(L.gv[q], ec[L.gi[q]], g);
  s = sum8(fma(-wd, s, g));
  if (on && t == 0) L.e[v] = fma(2.0 * wd, L.r[v], s);
}

// Levels tail .. nlev-1 as one matrix: block j runs their cycle (the last
// level by its inverse, or one sweep) on unit vector j, vectors in LDS, and
// writes row j of the symmetric result.  A solve applies it as often as it
// iterates: applying the levels in one workgroup took 17 us per iteration at
// 770 nodes, the matrix takes 5.
__global__ __launch_bounds__(256) void amg_dense_kernel(const AmgData* __restrict__ dA) {
  __shared__ double R[kAmgTailNodes], X[kAmgTailNodes];
  const AmgData& A = *dA;
  const int t0 = A.tail, last = A.nlev - 1, tid = threadIdx.x, n0 = A.lev[t0].n;
  for (int v = tid; v < n0; v += 256) R[v] = v == (int)blockIdx.x ? 1.0 : 0.0;
  __syncthreads();
  int o = 0;
  for (int l = t0; l < last; ++l) {
    const AmgLevel& L = A.lev[l];
    const int nc = A.lev[l + 1].n, on = o + L.n;
    for (int c = tid >> 3; c < nc; c += 32) {  // eight lanes per row, whole groups
      double s = 0.0;
      for (int t = L.tp[c] + (tid & 7); t < L.tp[c + 1]; t += 8) s = fma(L.gv[L.tx[t]], R[o + L.ti[t]], s);
      s = sum8(s);
      if ((tid & 7) == 0) R[on + c] = s;
    }
    o = on;
    __syncthreads();
  }
  const AmgLevel& Z = A.lev[last];
  for (int v = tid; v < Z.n; v += 256) {
    double s = 0.0;
    if (A.direct)
      for (int u = 0; u < Z.n; ++u) s = fma(A.cinv[u * Z.n + v], R[o + u], s);
    else
      s = Z.dinv[v] * R[o + v];
    X[o + v] = s;
  }
  __syncthreads();
  for (int l = last - 1; l >= t0; --l) {
    const AmgLevel& L = A.lev[l];
    const double* ec = X + o;
    o -= L.n;
    for (int v = tid; v < L.n; v += 256) {
      const double wd = L.dinv[v];
      double s = 0.0, g = 0.0;
      for (int e = L.ap[v]; e < L.ap[v + 1]; ++e) {
        const int w = L.ai[e];
        s = fma(L.av[e], L.dinv[w] * R[o + w], s);
      }
      for (int q = L.gp[v]; q < L.gp[v + 1]; ++q) g = fma(L.gv[q], ec[L.gi[q]], g);
      X[o + v] = wd * (2.0 * R[o + v] - s) + g;
    }
    __syncthreads();
  }
  for (int v = tid; v < n0; v += 256) A.dense[(size_t)blockIdx.x * n0 + v] = X[v];
}

// e = dense r on level tail: a wavefront per row.
__global__ __launch_bounds__(256) void amg_apply_kernel(const double* __restrict__ D, int n,
                                                        const double* __restrict__ r, double* __restrict__ e,
                                                        const CgState* st) {
  if (st->done) return;
  const int v = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (v >= n) return;
  double s = 0.0;
  for (int u = threadIdx.x & 63; u < n; u += 64) s = fma(D[(size_t)v * n + u], r[u], s);
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) e[v] = s;
}

// The last level on its own where it is too large for the tail: one sweep.
__global__ __launch_bounds__(256) void amg_sweep_kernel(AmgLevel L, const CgState* st) {
  if (st->done) return;
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v < L.n) L.e[v] = L.dinv[v] * L.r[v];
}

// z = t + G e, and the (r, z) partials the next product reads.
template <int NT>
__global__ __launch_bounds__(256) void amg_last_kernel(TraceSystem T, CgVectors v, AmgTop A) {
  __shared__ double sh[4];
  const CgState* st = v.st;
  if (st->done) return;
  const double* __restrict__ e = A.e;
  double p = 0.0;
  for (int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x; r < T.N; r += (int64_t)v.nblocks * 256) {
    const int4 u = *reinterpret_cast<const int4*>(A.fv + 4 * (r / NT));
    double z = A.t[r];
    z = fma(A.g[r], e[u.x], z);
    z = fma(A.g[T.N + r], e[u.y], z);
    z = fma(A.g[2 * T.N + r], e[max(u.z, 0)], z);  // G is zero where there is no vertex
    z = fma(A.g[3 * T.N + r], e[max(u.w, 0)], z);
    v.z[r] = z;
    p = fma(v.r[r], z, p);
  }
  p = wave_sum(p);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = p;
  __syncthreads();
  if (threadIdx.x == 0)
    v.part[(size_t)v.nblocks * (1 + (st->i_spmv & 1)) + blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

unsigned blocks_of(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

// --------------------------------------------------------------------- plan
using Ints = std::vector<int>;

// Greedy aggregation of a graph with self entries: a node whose neighbourhood
// is untouched founds an aggregate of it; nodes left over join a neighbour's.
int aggregate(int n, const Ints& ap, const Ints& ai, Ints& agg) {
  agg.assign(n, -1);
  int na = 0;
  for (int v = 0; v < n; ++v) {
    bool free = agg[v] < 0;
    for (int e = ap[v]; free && e < ap[v + 1]; ++e) free = agg[ai[e]] < 0;
    if (!free) continue;
    for (int e = ap[v]; e < ap[v + 1]; ++e) agg[ai[e]] = na;
    ++na;
  }
  Ints out = agg;
  for (int v = 0; v < n; ++v)
    for (int e = ap[v]; out[v] < 0 && e < ap[v + 1]; ++e) out[v] = agg[ai[e]];
  agg.swap(out);
  return na;
}

// Pattern of the product of two CSR patterns, rows sorted; false: more than
// 32-bit indices hold.
bool multiply(int n, const Ints& ap, const Ints& ai, const Ints& bp, const Ints& bi, int ncol, Ints& cp, Ints& ci) {
  Ints mark(ncol, -1);
  cp.assign(n + 1, 0);
  ci.clear();
  for (int v = 0; v < n; ++v) {
    for (int e = ap[v]; e < ap[v + 1]; ++e)
      for (int x = bp[ai[e]]; x < bp[ai[e] + 1]; ++x)
        if (mark[bi[x]] != v) {
          mark[bi[x]] = v;
          ci.push_back(bi[x]);
        }
    if (ci.size() > (size_t)INT32_MAX) return false;
    std::sort(ci.begin() + cp[v], ci.end());
    cp[v + 1] = (int)ci.size();
  }
  return true;
}

void transpose(int n, int ncol, const Ints& ap, const Ints& ai, Ints& tp, Ints& ti, Ints& tx) {
  tp.assign(ncol + 1, 0);
  for (int c : ai) ++tp[c + 1];
  for (int c = 0; c < ncol; ++c) tp[c + 1] += tp[c];
  ti.resize(ai.size());
  tx.resize(ai.size());
  Ints at(tp.begin(), tp.end() - 1);
  for (int v = 0; v < n; ++v)
    for (int e = ap[v]; e < ap[v + 1]; ++e) {
      const int k = at[ai[e]]++;
      ti[k] = v;
      tx[k] = e;
    }
}

}  // namespace

double amg_aspect(int64_t nc, const int* cn, const double* xy) {
  std::vector<double> a(nc);
  for (int64_t c = 0; c < nc; ++c) {
    double x[3], y[3], l2 = 0.0;
    for (int v = 0; v < 3; ++v) {
      const double *p = xy + 2 * (size_t)cn[3 * c + v], *q = xy + 2 * (size_t)cn[3 * c + (v + 1) % 3];
      x[v] = q[0] - p[0];
      y[v] = q[1] - p[1];
      l2 = std::max(l2, x[v] * x[v] + y[v] * y[v]);
    }
    const double twice = std::fabs(x[0] * y[1] - x[1] * y[0]);
    a[c] = l2 / (2.0 * twice);
    if (!(a[c] < HUGE_VAL)) a[c] = HUGE_VAL;  // no area, or no numbers
  }
  const int64_t q = nc * 3 / 4;
  std::nth_element(a.begin(), a.begin() + q, a.end());
  return a[q];
}

bool amg_plan(int64_t nn, int64_t nc, int64_t nf, const int* cn, const int* cf, const int* fcell, AmgPlan& plan) {
  plan = AmgPlan{};
  if (nn >= INT32_MAX / 8 || nf >= INT32_MAX / 8) return false;
  const int n = (int)nn;
  const auto put = [&](const Ints& v) {
    while (plan.ints.size() % 4) plan.ints.push_back(0);  // int4 reads
    const size_t at = plan.ints.size();
    plan.ints.insert(plan.ints.end(), v.begin(), v.end());
    return at;
  };
  // the vertices of every face; where a face's two cells name different nodes,
  // it joins them, lower end to lower end and higher to higher
  Ints fv(4 * nf, -1), to(n);
  for (int v = 0; v < n; ++v) to[v] = v;
  const auto vertex = [&](int v) {
    while (to[v] != v) v = to[v] = to[to[v]];
    return v;
  };
  for (int64_t f = 0; f < nf; ++f)
    for (int k = 0; k < 2; ++k) {
      const int64_t c = fcell[2 * f + k];
      if (c < 0) continue;
      const int l = cf[3 * c] == f ? 0 : (cf[3 * c + 1] == f ? 1 : (cf[3 * c + 2] == f ? 2 : -1));
      if (l < 0) return false;
      const int a = cn[3 * c + (l + 1) % 3], b = cn[3 * c + (l + 2) % 3], lo = std::min(a, b), hi = std::max(a, b);
      if (k == 0) {
        fv[4 * f] = lo;
        fv[4 * f + 1] = hi;
      } else if (fv[4 * f] != lo || fv[4 * f + 1] != hi) {
        to[vertex(lo)] = vertex(fv[4 * f]);
        to[vertex(hi)] = vertex(fv[4 * f + 1]);
        plan.joined = true;
      }
      fv[4 * f + 2 + k] = cn[3 * c + l];
    }
  if (plan.joined) {
    Ints cv(3 * nc);
    for (int64_t i = 0; i < 3 * nc; ++i) cv[i] = vertex(cn[i]);
    for (int64_t c = 0; c < nc; ++c)  // a cell across the whole mesh
      if (cv[3 * c] == cv[3 * c + 1] || cv[3 * c + 1] == cv[3 * c + 2] || cv[3 * c + 2] == cv[3 * c]) return false;
    for (int64_t f = 0; f < nf; ++f) {
      for (int j = 0; j < 4; ++j)
        if (fv[4 * f + j] >= 0) fv[4 * f + j] = vertex(fv[4 * f + j]);
      if (fv[4 * f + 2] == fv[4 * f + 3]) return false;  // two cells across it
    }
    plan.cv = put(cv);
  }
  // the faces of every vertex
  Ints vp(n + 1, 0), vi;
  for (int v : fv)
    if (v >= 0) ++vp[v + 1];
  for (int v = 0; v < n; ++v) vp[v + 1] += vp[v];
  vi.resize(vp[n]);
  {
    Ints at(vp.begin(), vp.end() - 1);
    for (int64_t u = 0; u < 4 * nf; ++u)
      if (fv[u] >= 0) vi[at[fv[u]]++] = (int)u;
  }
  // the vertex graph: each vertex, then the other ends of its faces, sorted
  Ints ap(n + 1, 0), ai, af;
  std::vector<std::pair<int, int>> row;
  for (int v = 0; v < n; ++v) {
    row.assign(1, {v, -1});
    for (int e = vp[v]; e < vp[v + 1]; ++e)
      if ((vi[e] & 3) < 2) row.push_back({fv[vi[e] ^ 1], vi[e] >> 2});
    std::sort(row.begin(), row.end());
    for (const auto& [w, f] : row) {
      ai.push_back(w);
      af.push_back(f);
    }
    ap[v + 1] = (int)ai.size();
  }
  plan.fv = put(fv);
  plan.vp = put(vp);
  plan.vi = put(vi);
  plan.af = put(af);
  int nl = n;
  for (int l = 0;; ++l) {
    AmgPlan::Level& L = plan.lev[l];
    L.n = nl;
    L.nnz = (int)ai.size();
    L.ap = put(ap);
    L.ai = put(ai);
    plan.nlev = l + 1;
    plan.direct = nl <= kAmgDirect;
    if (plan.direct || l + 1 == kAmgLevels) break;
    Ints agg, idp(nl + 1), pp, pi, gp, gi, tp, ti, tx, xp, xi;
    const int na = aggregate(nl, ap, ai, agg);
    if (na > nl * 0.8) break;
    for (int v = 0; v <= nl; ++v) idp[v] = v;
    if (!multiply(nl, ap, ai, idp, agg, na, pp, pi) || !multiply(nl, ap, ai, pp, pi, na, gp, gi)) return false;
    transpose(nl, na, pp, pi, tp, ti, tx);
    if (!multiply(na, tp, ti, gp, gi, na, xp, xi)) return false;
    transpose(nl, na, gp, gi, tp, ti, tx);
    L.gnnz = (int)gi.size();
    L.agg = put(agg);
    L.gp = put(gp);
    L.gi = put(gi);
    L.tp = put(tp);
    L.ti = put(ti);
    L.tx = put(tx);
    ap.swap(xp);
    ai.swap(xi);
    nl = na;
  }
  // smallest suffix of levels within the matrix's budget
  plan.tail = plan.nlev;
  int64_t nodes = 0;
  for (int l = plan.nlev - 1; l >= 0; --l) {
    nodes += plan.lev[l].n;
    if (nodes > kAmgTailNodes || plan.lev[l].n > kAmgDense) break;
    plan.tail = l;
  }
  return true;
}

int launch_amg_setup(const DevMesh& m, const TraceSystem& T, const double* Ate, const AmgData& A, const AmgData* dA,
                     hipStream_t s) {
  const int n = A.lev[0].n;
  hipLaunchKernelGGL(amg_fix_kernel, dim3(blocks_of(n, 256)), dim3(256), 0, s, A.top, T);
  hipLaunchKernelGGL(amg_vertex_kernel, dim3(blocks_of(n, 32)), dim3(256), 0, s, m, T.nt, Ate, A.top, A.lev[0]);
#define GK(NT)                                                                                                       \
  case NT:                                                                                                           \
    hipLaunchKernelGGL(amg_g_kernel<NT>, dim3(blocks_of(T.N, 64 * NT)), dim3(64 * NT), 0, s, m, T, Ate, A.top);      \
    break;
  switch (T.nt) { GK(2) GK(3) GK(4) GK(5) }
#undef GK
  for (int l = 0; l < A.nlev; ++l) {
    const AmgLevel& L = A.lev[l];
    const bool last = l + 1 == A.nlev;
    if (last && A.direct) {
      hipLaunchKernelGGL(amg_inverse_kernel, dim3(1), dim3(256), 0, s, L, A.cinv);
      break;
    }
    hipLaunchKernelGGL(amg_p_kernel, dim3(blocks_of(L.n, 32)), dim3(256), 0, s, L, last ? 0 : 1);
    if (last) break;
    hipLaunchKernelGGL(amg_ap_kernel, dim3(blocks_of(L.n, 32)), dim3(256), 0, s, L);
    hipLaunchKernelGGL(amg_rap_kernel, dim3(A.lev[l + 1].n), dim3(256), 0, s, L, A.lev[l + 1]);
  }
  if (A.tail < A.nlev) hipLaunchKernelGGL(amg_dense_kernel, dim3(A.lev[A.tail].n), dim3(256), 0, s, dA);
  return (int)hipGetLastError();
}

int launch_amg_cycle(const DevPattern& P, const TraceSystem& T, const CgVectors& cg, const AmgData& A,
                     double rtol2, int maxit, hipStream_t s) {
  if (!trace_op_ready(P, T)) return (int)hipErrorInvalidValue;
  const int nbv = (int)blocks_of(A.lev[0].n, 8 * T.nt);
#define FK(NT)                                                                                                       \
  case NT:                                                                                                           \
    hipLaunchKernelGGL(amg_first_kernel<NT>, dim3(nbv + blocks_of(T.N, 64 * NT)), dim3(64 * NT), 0, s, P, T, cg,     \
                       A.top, nbv, rtol2, maxit);                                                                          \
    break;
  switch (T.nt) { FK(2) FK(3) FK(4) FK(5) }
#undef FK
  const int down = std::min(A.tail, A.nlev - 1);
  for (int l = 0; l < down; ++l)
    hipLaunchKernelGGL(amg_restrict_kernel, dim3(blocks_of(A.lev[l + 1].n, 16)), dim3(256), 0, s, A.lev[l],
                       A.lev[l + 1], cg.st);
  if (A.tail < A.nlev)
    hipLaunchKernelGGL(amg_apply_kernel, dim3(blocks_of(A.lev[down].n, 4)), dim3(256), 0, s, A.dense, A.lev[down].n,
                       A.lev[down].r, A.lev[down].e, cg.st);
  else
    hipLaunchKernelGGL(amg_sweep_kernel, dim3(blocks_of(A.lev[down].n, 256)), dim3(256), 0, s, A.lev[down], cg.st);
  for (int l = down - 1; l >= 0; --l)
    hipLaunchKernelGGL(amg_post_kernel, dim3(blocks_of(A.lev[l].n, 32)), dim3(256), 0, s, A.lev[l], A.lev[l + 1].e,
                       cg.st);
#define LK(NT)                                                                                        \
  case NT:                                                                                            \
    hipLaunchKernelGGL(amg_last_kernel<NT>, dim3(cg.nblocks), dim3(256), 0, s, T, cg, A.top);         \
    break;
  switch (T.nt) { LK(2) LK(3) LK(4) LK(5) }
#undef LK
  return (int)hipGetLastError();
}

}  // namespace hdg
