// The reduced trace system of rectangle meshes: set-up and CG kernels.  See
// hdg_quad.h for the system and the layout.
//
// One CG iteration i:
//   product(i):  convergence test, beta; q = T z + beta q, p = z + beta p; (p, q)
//   residual(i): alpha; x += alpha p, r -= alpha q; e0 = omega Dinv r (not
//                stored); res = r - T e0; (r, r); r1 = P^T res
//   V-cycle on the vertices: e1
//   smooth(i):   z = P e1 + omega Dinv (r + res - (T P) e1); (r, z)
// so the matrix is read twice per iteration.  r alternates between two
// buffers (a neighbour's r and q are read while the point's own r is
// written).  Every sum over a row is formed in a fixed order that does not
// depend on the launch partition, and every reduction over an instance's own
// blocks, so an instance gets the same bits alone and in a group.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "hdg_quad.h"

namespace hdg {

namespace {

constexpr double kS3 = 0.28867513459481288225;  // 1 / (2 sqrt 3)
constexpr int kNW = kQuadThreads / 64;

struct SelOne {
  QuadInst I;
};
struct SelGroup {
  const QuadInst* inst;
  const BlockMap* map;
};
__device__ __forceinline__ const QuadInst& inst_of(const SelOne& s, int& lb) {
  lb = blockIdx.x;
  return s.I;
}
__device__ __forceinline__ const QuadInst& inst_of(const SelGroup& s, int& lb) {
  const BlockMap m = s.map[blockIdx.x];
  lb = m.lb;
  return s.inst[m.inst];
}
// one block per instance
__device__ __forceinline__ const QuadInst& inst_block(const SelOne& s) { return s.I; }
__device__ __forceinline__ const QuadInst& inst_block(const SelGroup& s) { return s.inst[blockIdx.x]; }

// offset of value 0 of point g in an array with NS values per point
template <int NS>
__device__ __forceinline__ int64_t at(const QuadInst& I, int g) {
  return (I.tile0 + (g >> 6)) * (int64_t)(NS * 64) + (g & 63);
}

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}
__device__ __forceinline__ double bsum(double v, double* sh) {
  v = wsum(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) sh[w] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < kNW; ++i) s += sh[i];
  __syncthreads();
  return s;
}
__device__ __forceinline__ double psum(const double* p, int n, double* sh) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kQuadThreads) s += p[i];
  return bsum(s, sh);
}
// A thread's share of n partials, loaded ahead of whatever follows: the CG
// kernels read the solve's state and the partials of the kernel before them
// in one flight and branch on `done` afterwards (each read is a trip to memory
// past the XCD's own L2 and most of a small problem's kernel time: 32^2 P1
// product 6.5 -> 6.4 us, residual 8.3 -> 7.9).
__device__ __forceinline__ double pshare(const double* p, int n) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kQuadThreads) s += p[i];
  asm volatile("" : "+v"(s));
  return s;
}

// entry (a, b) of a triangle
__device__ __forceinline__ constexpr int tri(int nt, int a, int b) { return dinv_slot(nt, a, b); }

// faces of a grid point in the natural numbering (0-based)
__device__ __forceinline__ int face_h(const QuadSys& S, const QuadInst& I, int i, int j) {
  return j < I.ny ? S.cf[3 * (I.cell0 + 2 * ((int64_t)j * I.nx + i)) + 2]
                  : S.cf[3 * (I.cell0 + 2 * ((int64_t)(I.ny - 1) * I.nx + i) + 1)];
}
__device__ __forceinline__ int face_v(const QuadSys& S, const QuadInst& I, int i, int j) {
  return i < I.nx ? S.cf[3 * (I.cell0 + 2 * ((int64_t)j * I.nx + i)) + 1]
                  : S.cf[3 * (I.cell0 + 2 * ((int64_t)j * I.nx + I.nx - 1) + 1) + 2];
}
__device__ __forceinline__ int face_d(const QuadSys& S, const QuadInst& I, int i, int j) {
  return S.cf[3 * (I.cell0 + 2 * ((int64_t)j * I.nx + i))];
}

// ---------------------------------------------------------------- set-up
// Dof masks of the axis faces; a vertex is fixed when a face through it has
// a prescribed mode-0 dof.  *I.plain: a diagonal face has a prescribed dof.
template <class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_mask_kernel(QuadSys S, Sel sel) {
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  const int nt = S.nt;
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.ntiles * 64; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W;
    unsigned m = 0;
    unsigned char fix = 0;
    const bool in = g < I.G;
    if (in && i < I.nx) {
      const int64_t f = (int64_t)face_h(S, I, i, j) * nt;
      for (int a = 0; a < nt; ++a) m |= (S.dmask[f + a] ? 1u : 0u) << a;
    } else {
      m |= (1u << nt) - 1;
    }
    if (in && j < I.ny) {
      const int64_t f = (int64_t)face_v(S, I, i, j) * nt;
      for (int a = 0; a < nt; ++a) m |= (S.dmask[f + a] ? 1u : 0u) << (nt + a);
    } else {
      m |= ((1u << nt) - 1) << nt;
    }
    S.mask[(I.tile0 << 6) + g] = (unsigned short)m;
    if (!in) continue;
    if (i < I.nx) fix |= m & 1;
    if (j < I.ny) fix |= (m >> nt) & 1;
    if (i > 0) fix |= S.dmask[(int64_t)face_h(S, I, i - 1, j) * nt];
    if (j > 0) fix |= S.dmask[(int64_t)face_v(S, I, i, j - 1) * nt];
    if (i > 0 && j < I.ny) fix |= S.dmask[(int64_t)face_d(S, I, i - 1, j) * nt];
    if (i < I.nx && j > 0) fix |= S.dmask[(int64_t)face_d(S, I, i, j - 1) * nt];
    I.vmask[g] = fix ? 1 : 0;
    if (i < I.nx && j < I.ny) {
      const int64_t f = (int64_t)face_d(S, I, i, j) * nt;
      for (int a = 0; a < nt; ++a)
        if (S.dmask[f + a]) *I.plain = 1;
    }
  }
}

// Zero couplings at the points without a quad (the last column and row, the end
// of the last tile); the set-up writes all others.  (A memset of the whole array
// was 0.16 of the 0.9 ms of hdg_setup at 1024^2 P3.)
template <class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_clear_kernel(QuadSys S, Sel sel) {
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  const int ns = quad_blk_vals(S.nt);
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.ntiles * 64; g += I.nbE * kQuadThreads) {
    if (g < I.G && g % I.W < I.nx && g / I.W < I.ny) continue;
    double* b = S.blk + (I.tile0 + (g >> 6)) * (int64_t)(ns * 64) + (g & 63);
    for (int s = 0; s < ns; ++s) b[s * 64] = 0.0;
  }
}

// Lanes per quad of the set-up kernels (one per column of the quad's 4 nt
// axis dofs) and quads per block.
constexpr int lanes_per_quad(int nt) { return nt == 2 ? 8 : (nt <= 4 ? 16 : 32); }
constexpr int quads_per_block(int nt) { return kQuadThreads / lanes_per_quad(nt); }
// Stride of a quad's two staged cell blocks: the lanes of a quad read
// neighbouring columns, so the quads of a wavefront are set 8 (two modes) or
// 16 doubles apart modulo the 32 of an LDS row (unpadded, 288 doubles at four
// modes put them all in the same banks).
constexpr int quad_stride(int nt) {
  const int n = 18 * nt * nt, want = nt == 2 ? 8 : 16;
  return n + ((want - n) % 32 + 32) % 32;
}

// entry K[(f, a), (g, b)] of the assembled matrix, rounded to float
template <int NT>
__device__ double k_entry(const QuadSys& S, int64_t f, int a, int64_t g, int b) {
  if constexpr (kSymBlocks<NT>) {
    const int64_t nf = S.K.nf;
    if (f == g) return (double)(float)S.K.blk[(int64_t)dinv_slot(NT, a, b) * nf + f];
    const double* own = S.K.blk + (int64_t)(NT * (NT + 1) / 2) * nf;
    for (int k = 0; k < 2; ++k) {
      if (S.P.nbr[4 * f + k] == g) return (double)(float)own[((2 * f + k) * NT + a) * NT + b];
      const int code = S.P.nbr[4 * f + 2 + k];
      if ((code >> 1) == g) return (double)(float)own[((2 * g + (code & 1)) * NT + b) * NT + a];
    }
    return 0.0;
  } else {
    for (int s = 0; s < S.P.nslot[f]; ++s)
      if (S.P.bcol[f * kSlots + s] == g) return (double)(float)S.K.vals[(int64_t)(s * NT + b) * S.K.N + f * NT + a];
    return 0.0;
  }
}

// The two cells' condensed blocks and loads of the block's quads on their way
// to LDS, A[quad][cell][row][column], b[quad][cell][row] (quads q0 .. q0 + nq - 1): every
// load (and the kernel's own) is issued before the first is stored.  With a
// loop of loads and stores the set-up was bound by that latency (1024^2 P3 2.4
// ms, now 1.5; 768^2 P1 0.31, now 0.21; finish 1.06, now 0.80); several groups
// per block, the next fetched ahead, took more registers than it hid (2.9 ms).
template <int NT>
struct CellFetch {
  static constexpr int CA = 9 * NT * NT, NTR = 3 * NT, QB = quads_per_block(NT);
  static constexpr int NA = (QB * CA + kQuadThreads - 1) / kQuadThreads;
  static constexpr int NL = (QB * 2 * NTR + kQuadThreads - 1) / kQuadThreads;
  typedef double V2 __attribute__((ext_vector_type(2)));
  V2 va[NA];
  double vb[NL];
  __device__ __forceinline__ void fetch(const QuadSys& S, const QuadInst& I, int q0, int nq) {
    const V2* s2 = reinterpret_cast<const V2*>(S.Ate + (I.cell0 + 2 * (int64_t)q0) * CA);
    const double* sb = S.bte + (I.cell0 + 2 * (int64_t)q0) * NTR;
#pragma unroll
    for (int k = 0; k < NA; ++k) va[k] = s2[min((int)threadIdx.x + kQuadThreads * k, nq * CA - 1)];
#pragma unroll
    for (int k = 0; k < NL; ++k) vb[k] = sb[min((int)threadIdx.x + kQuadThreads * k, nq * 2 * NTR - 1)];
  }
  __device__ __forceinline__ void stage(double* A, double* b, int nq) const {
    constexpr int QS = quad_stride(NT);
    V2* d2 = reinterpret_cast<V2*>(A);
#pragma unroll
    for (int k = 0; k < NA; ++k) {
      const int e = threadIdx.x + kQuadThreads * k;
      if (e < nq * CA) d2[(e / CA) * (QS / 2) + e % CA] = va[k];
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int e = threadIdx.x + kQuadThreads * k;
      if (e < nq * 2 * NTR) b[e] = vb[k];
    }
  }
};

// The same from the assembled matrix (S.from_k): K_DD, the couplings and the
// loads split between the two cells, the axis faces' own blocks left zero
// (q_diag_kernel adds them).
template <int NT>
__device__ __forceinline__ void stage_assembled(const QuadSys& S, const QuadInst& I, int q0, int nq, double* A,
                                                double* b) {
  constexpr int NTR = 3 * NT, CA = NTR * NTR, QS = quad_stride(NT);
  for (int e = threadIdx.x; e < nq * 2 * CA; e += kQuadThreads) {
    const int q = q0 + e / (2 * CA), cell = (e / CA) & 1, r = (e % CA) / NTR, c = e % NTR;
    const int lr = r / NT, lc = c / NT, ld = cell;  // local face of D: 0 below, 1 above
    const int64_t c3 = 3 * (I.cell0 + 2 * (int64_t)q + cell);
    double v = 0.0;
    if (lr != lc || (lr == ld && cell == 0)) v = k_entry<NT>(S, S.cf[c3 + lr], r % NT, S.cf[c3 + lc], c % NT);
    A[(e / (2 * CA)) * QS + e % (2 * CA)] = v;
  }
  for (int e = threadIdx.x; e < nq * 2 * NTR; e += kQuadThreads) {
    const int q = q0 + e / (2 * NTR), cell = (e / NTR) & 1, r = e % NTR, lr = r / NT;
    const int i = q % I.nx, j = q / I.nx;
    const int64_t f = S.cf[3 * (I.cell0 + 2 * (int64_t)q + cell) + lr];
    const bool mine = cell == 0 || (lr == 0 && j == I.ny - 1) || (lr == 2 && i == I.nx - 1);
    b[e] = mine ? S.K.rhs[f * NT + r % NT] : 0.0;
  }
}

// LDL^T of S_DD = -(K_DD) on the free dofs of D (identity rows on the
// prescribed ones): unit lower factor l, reciprocal pivots.
template <int NT>
struct DiagFactor {
  double l[NT][NT], di[NT];
};
template <int NT, class M>
__device__ __forceinline__ DiagFactor<NT> factor_d(const double* Al, const double* Au, const M& masked) {
  constexpr int NTR = 3 * NT;
  DiagFactor<NT> F;
  double d[NT];
#pragma unroll
  for (int a = 0; a < NT; ++a) {
#pragma unroll
    for (int b = 0; b <= a; ++b) {
      const bool mk = masked(a) || masked(b);
      double v = mk ? (a == b ? 1.0 : 0.0) : -(Al[a * NTR + b] + Au[(NT + a) * NTR + NT + b]);
#pragma unroll
      for (int k = 0; k < b; ++k) v = fma(-F.l[a][k] * d[k], F.l[b][k], v);
      if (a == b) {
        d[a] = v;
        F.di[a] = 1.0 / v;
      } else {
        F.l[a][b] = v * F.di[b];
      }
    }
  }
  return F;
}

// The quads' systems.  One lane per column c = (face f, mode b) of a quad's
// 4 nt axis dofs (f = B, T, L, R): T_Q = S_oo - S_oD S_DD^-1 S_Do with the
// cells' blocks staged in LDS by 16-byte loads, the couplings, the diagonal
// parts and the loads written through LDS in runs of one value over the
// block's consecutive quads.  HBM-bound: it reads the condensed blocks once
// (2 (3nt)^2 doubles per quad) and writes 6 nt^2 + 2 nt (nt+1) + 9 nt + 10.
template <int NT, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_build_kernel(QuadSys S, Sel sel) {
  constexpr int NTR = 3 * NT, CA = NTR * NTR, LPQ = lanes_per_quad(NT), QB = quads_per_block(NT);
  constexpr int NB = NT * NT, NS = NT * (NT + 1) / 2, NC = 4 * NT;
  constexpr int kOut = 6 * NB + 4 * NS + 9 * NT + kQuadCq;
  constexpr int QS = quad_stride(NT), WS = NT * NC + 2, OS = QB + 1;
  static_assert(kOut * OS <= QB * QS, "the output staging reuses the cells' blocks");
  __shared__ double A[QB * QS];
  __shared__ double bs[QB * 2 * NTR], us[QB * 2 * NTR];
  __shared__ double Ws[QB * WS];
  __shared__ int gq[QB];
  __shared__ double Ps[QB * 8 * 4];
  __shared__ unsigned char ms[QB * 2 * NTR];
  __shared__ int lift[QB];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  const int nquads = I.nx * I.ny;
  const int q0 = lb * QB, nq = min(QB, nquads - q0);
  // dofs of the quads' faces and their masks, fetched beside the cells' blocks
  constexpr int NM = (QB * 2 * NTR + kQuadThreads - 1) / kQuadThreads;
  CellFetch<NT> cells;
  int64_t fd[NM];
  unsigned char md[NM];
#pragma unroll
  for (int k = 0; k < NM; ++k) {
    const int e = min((int)threadIdx.x + kQuadThreads * k, nq * 2 * NTR - 1), r = e % NTR;
    fd[k] = (int64_t)S.cf[3 * (I.cell0 + 2 * (int64_t)q0 + e / NTR) + r / NT] * NT + r % NT;
  }
#pragma unroll
  for (int k = 0; k < NM; ++k) md[k] = S.dmask[fd[k]];
  if (!S.from_k) cells.fetch(S, I, q0, nq);
  if (threadIdx.x < QB) {
    const int q = q0 + min((int)threadIdx.x, nq - 1);
    lift[threadIdx.x] = 0;
    gq[threadIdx.x] = (q / I.nx) * I.W + q % I.nx;
  }
  if (S.from_k)
    stage_assembled<NT>(S, I, q0, nq, A, bs);
  else
    cells.stage(A, bs, nq);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NM; ++k) {
    const int e = threadIdx.x + kQuadThreads * k;
    const double u = md[k] ? S.uD[fd[k]] : 0.0;
    if (e >= nq * 2 * NTR) continue;
    ms[e] = md[k];
    us[e] = u;
    if (u != 0.0) lift[e / (2 * NTR)] = 1;
  }
  __syncthreads();
  const int ql = threadIdx.x / LPQ, c = threadIdx.x % LPQ;
  const bool live = ql < nq && c < NC;
  const int f = c / NT, b = c - f * NT;
  // cell and local face of B, T, L, R
  const int cell = f & 1, lf = f == 0 ? 2 : (f == 1 ? 0 : (f == 2 ? 1 : 2));
  const double* Al = A + ql * QS;
  const double* Au = Al + CA;
  double Tc[NC], w[NT], bD[NT], bred = 0.0, braw = 0.0, tpq[4] = {0, 0, 0, 0};
  if (live) {
    const double* Ac = cell ? Au : Al;
    const double* bc = bs + ql * 2 * NTR + cell * NTR;
    const double* uc = us + ql * 2 * NTR + cell * NTR;
    const unsigned char* mD = ms + ql * 2 * NTR;  // D is local face 0 of the lower cell
    const int col = lf * NT + b, dr = cell * NT;  // D rows of this column's cell
    auto masked = [&](int a) { return mD[a] != 0; };
    const DiagFactor<NT> F = factor_d<NT>(Al, Au, masked);
    // w = l^-1 S_D,c and the D load
    const double* bl = bs + ql * 2 * NTR;
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      double s = masked(a) ? 0.0 : -Ac[(dr + a) * NTR + col];
      double t = -(bl[a] + bl[NTR + NT + a]);
      if (lift[ql]) {
        const double* ul = us + ql * 2 * NTR;
        for (int k = 0; k < NTR; ++k) t = fma(Al[a * NTR + k], ul[k], t);
        for (int k = 0; k < NTR; ++k) t = fma(Au[(NT + a) * NTR + k], ul[NTR + k], t);
      }
      bD[a] = masked(a) ? 0.0 : t;
#pragma unroll
      for (int k = 0; k < a; ++k) s = fma(-F.l[a][k], w[k], s);
      w[a] = s;
    }
    double y[NT];
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      double t = bD[a];
#pragma unroll
      for (int k = 0; k < a; ++k) t = fma(-F.l[a][k], y[k], t);
      y[a] = t;
    }
    braw = -bc[col];
    if (lift[ql])
      for (int k = 0; k < NTR; ++k) braw = fma(Ac[col * NTR + k], uc[k], braw);
    bred = braw;
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      bred = fma(-w[a], y[a] * F.di[a], bred);
      Ws[ql * WS + a * NC + c] = w[a];
      w[a] *= F.di[a];
    }
    // the cell's own part of the column: rows of the faces of the same cell
#pragma unroll
    for (int r = 0; r < NC; ++r) {
      const int fr = r / NT, lr = fr == 0 ? 2 : (fr == 1 ? 0 : (fr == 2 ? 1 : 2));
      Tc[r] = (fr & 1) == cell ? -Ac[(lr * NT + r - fr * NT) * NTR + col] : 0.0;
    }
  }
  __syncthreads();
  if (live) {
#pragma unroll
    for (int r = 0; r < NC; ++r) {
      double t = Tc[r];
#pragma unroll
      for (int a = 0; a < NT; ++a) t = fma(-Ws[ql * WS + a * NC + r], w[a], t);
      Tc[r] = t;
    }
    // row c of T P on the quad's vertices (i,j), (i+1,j), (i,j+1), (i+1,j+1),
    // prescribed dofs and fixed vertices left out
    if (b < 2) {
      const int v0 = gq[ql];
      const double keep[4] = {I.vmask[v0] ? 0.0 : 1.0, I.vmask[v0 + 1] ? 0.0 : 1.0, I.vmask[v0 + I.W] ? 0.0 : 1.0,
                              I.vmask[v0 + I.W + 1] ? 0.0 : 1.0};
      const unsigned char* mq = ms + ql * 2 * NTR;
#pragma unroll
      for (int fr = 0; fr < 4; ++fr) {
        const int lr = fr == 0 ? 2 : (fr == 1 ? 0 : (fr == 2 ? 1 : 2));
        const int lo = fr == 0 ? 0 : (fr == 1 ? 2 : (fr == 2 ? 0 : 1)), hi = fr == 0 ? 1 : (fr == 1 ? 3 : (fr == 2 ? 2 : 3));
        const unsigned char* mf = mq + (fr & 1) * NTR + lr * NT;
        const double t0 = mf[0] ? 0.0 : 0.5 * Tc[fr * NT], t1 = mf[1] ? 0.0 : kS3 * Tc[fr * NT + 1];
        tpq[lo] = fma(keep[lo], t0 - t1, tpq[lo]);
        tpq[hi] = fma(keep[hi], t0 + t1, tpq[hi]);
      }
      double* pr = Ps + (ql * 8 + f * 2 + b) * 4;
#pragma unroll
      for (int v = 0; v < 4; ++v) pr[v] = tpq[v];
    }
  }
  __syncthreads();
  // outputs, value-major over the block's quads, in the LDS of the blocks
  double* const O = A;
  auto put = [&](int s, double v) { O[s * OS + ql] = v; };
  if (live) {
    // couplings (row face, column face) BT LR BL BR TL TR
#pragma unroll
    for (int r = 0; r < NC; ++r) {
      const int fr = r / NT, a = r - fr * NT;
      if (fr < f) {
        // pair index of (fr, f)
        const int pair = fr == 0 ? (f == 1 ? 0 : (f == 2 ? 2 : 3)) : (fr == 1 ? (f == 2 ? 4 : 5) : 1);
        put(pair * NB + a * NT + b, Tc[r]);
      } else if (fr == f && a <= b) {
        put(6 * NB + f * NS + tri(NT, a, b), Tc[r]);
      }
    }
    const int ob = 6 * NB + 4 * NS;
    put(ob + c, bred);
    put(ob + NC + c, braw);
    if (c < NT) {
      double t = 0.0;
#pragma unroll
      for (int a = 0; a < NT; ++a) t = a == c ? bD[a] : t;
      put(ob + 2 * NC + c, t);
    }
  }
  // P^T (T P): 10 entries per quad
  for (int e = threadIdx.x; e < nq * kQuadCq; e += kQuadThreads) {
    const int qe = e / kQuadCq, t = e % kQuadCq;
    const int u = t < 4 ? 0 : (t < 7 ? 1 : (t < 9 ? 2 : 3)), v = t < 4 ? t : (t < 7 ? t - 3 : (t < 9 ? t - 5 : 3));
    const int vx = gq[qe] + (u >> 1) * I.W + (u & 1);
    double s = 0.0;
    for (int fr = 0; fr < 4; ++fr) {
      const int lr = fr == 0 ? 2 : (fr == 1 ? 0 : (fr == 2 ? 1 : 2));
      const int lo = fr == 0 ? 0 : (fr == 1 ? 2 : (fr == 2 ? 0 : 1)), hi = fr == 0 ? 1 : (fr == 1 ? 3 : (fr == 2 ? 2 : 3));
      if (u != lo && u != hi) continue;
      const unsigned char* mf = ms + qe * 2 * NTR + (fr & 1) * NTR + lr * NT;
      const double* pr = Ps + (qe * 8 + fr * 2) * 4;
      if (!mf[0]) s = fma(0.5, pr[v], s);
      if (!mf[1]) s = fma(u == hi ? kS3 : -kS3, pr[4 + v], s);
    }
    O[(6 * NB + 4 * NS + 9 * NT + t) * OS + qe] = I.vmask[vx] ? 0.0 : s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kOut * QB; e += kQuadThreads) {
    const int s = e / QB, qe = e % QB;
    if (qe >= nq) continue;
    const int g = gq[qe];
    const double v = O[s * OS + qe];
    if (s < 6 * NB)
      S.blk[at<6 * NB>(I, g) + s * 64] = v;
    else if (s < 6 * NB + 4 * NS)
      S.tp[at<12 * NT>(I, g) + (s - 6 * NB) * 64] = v;
    else if (s < 6 * NB + 4 * NS + 9 * NT)
      S.bq[at<9 * NT>(I, g) + (s - 6 * NB - 4 * NS) * 64] = v;
    else
      S.cq[at<kQuadCq>(I, g) + (s - 6 * NB - 4 * NS - 9 * NT) * 64] = v;
  }
}

// inverse of the symmetric a (upper triangle) with identity rows on the
// masked dofs, zero there in the result; by LDL^T
template <int NT>
__device__ __forceinline__ void inverse_masked(const double* a, unsigned m, double* inv) {
  double l[NT][NT], d[NT], di[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j <= i; ++j) {
      const bool mk = ((m >> i) | (m >> j)) & 1;
      double v = mk ? (i == j ? 1.0 : 0.0) : a[tri(NT, j, i)];
#pragma unroll
      for (int k = 0; k < j; ++k) v = fma(-l[i][k] * d[k], l[j][k], v);
      if (i == j) {
        d[i] = v;
        di[i] = 1.0 / v;
      } else {
        l[i][j] = v * di[j];
      }
    }
  // columns of l^-1, then sum of w_k di_k w_k^T
  double li[NT][NT];
#pragma unroll
  for (int c = 0; c < NT; ++c)
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      double v = i == c ? 1.0 : 0.0;
#pragma unroll
      for (int k = 0; k < i; ++k)
        if (k >= c) v = fma(-l[i][k], li[k][c], v);
      li[i][c] = i < c ? 0.0 : v;
    }
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = i; j < NT; ++j) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < NT; ++k)
        if (k >= j) v = fma(li[k][i] * di[k], li[k][j], v);
      inv[tri(NT, i, j)] = ((m >> i) | (m >> j)) & 1 ? 0.0 : v;
    }
}

// diagonal blocks (the two quads' parts) and their inverses
template <int NT, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_diag_kernel(QuadSys S, Sel sel) {
  constexpr int NS = NT * (NT + 1) / 2;
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.G; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W;
    const unsigned m = S.mask[(I.tile0 << 6) + g];
    const bool quad = i < I.nx && j < I.ny;
    double d[NS], inv[NS];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      // H: B of quad (i, j) and T of (i, j-1); V: L of (i, j) and R of (i-1, j)
      const bool other = f == 0 ? (j > 0 && i < I.nx) : (i > 0 && j < I.ny);
      const double* own = S.tp + at<12 * NT>(I, g) + (2 * f) * NS * 64;
      const double* oth = S.tp + at<12 * NT>(I, other ? (f == 0 ? g - I.W : g - 1) : g) + (2 * f + 1) * NS * 64;
      const bool exists = f == 0 ? i < I.nx : j < I.ny;
#pragma unroll
      for (int s = 0; s < NS; ++s) d[s] = (quad ? own[s * 64] : 0.0) + (other ? oth[s * 64] : 0.0);
      if (S.from_k && exists) {
        const int64_t fc = f == 0 ? face_h(S, I, i, j) : face_v(S, I, i, j);
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
          for (int b = a; b < NT; ++b) d[tri(NT, a, b)] -= k_entry<NT>(S, fc, a, fc, b);
      }
      inverse_masked<NT>(d, (m >> (f * NT)) & ((1u << NT) - 1), inv);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        S.D[at<2 * NS>(I, g) + (f * NS + s) * 64] = d[s];
        S.Dinv[at<2 * NS>(I, g) + (f * NS + s) * 64] = inv[s];
      }
    }
  }
}

// T P rows of the axis faces (hdg_quad.h): H(i, j) on the vertices (i,j),
// (i+1,j), (i,j+1), (i+1,j+1), (i,j-1), (i+1,j-1); V(i, j) on (i,j), (i,j+1),
// (i+1,j), (i+1,j+1), (i-1,j), (i-1,j+1).  Columns of fixed vertices are left
// in (e1 is zero there).
template <int NT, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_tp_kernel(QuadSys S, Sel sel) {
  constexpr int NB = NT * NT, NS = NT * (NT + 1) / 2;
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.G; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W;
    const unsigned short* mk = S.mask + (I.tile0 << 6);
    const bool quad = i < I.nx && j < I.ny, below = j > 0 && i < I.nx, left = i > 0 && j < I.ny;
    const unsigned m = mk[g], mu = j < I.ny ? mk[g + I.W] : ~0u, mr = i < I.nx ? mk[g + 1] : ~0u;
    const unsigned md = j > 0 ? mk[g - I.W] : ~0u, mdr = below ? mk[g - I.W + 1] : ~0u;
    const unsigned ml = i > 0 ? mk[g - 1] : ~0u, mlu = left ? mk[g - 1 + I.W] : ~0u;
    const double* bo = S.blk + at<6 * NB>(I, g);
    const double* bd = S.blk + at<6 * NB>(I, below ? g - I.W : g);
    const double* bl = S.blk + at<6 * NB>(I, left ? g - 1 : g);
    const double* dd = S.D + at<2 * NS>(I, g);
    double* out = S.tp + at<12 * NT>(I, g);
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      double t[6] = {0, 0, 0, 0, 0, 0};
      // columns 0 and 1 of a neighbour's block, on its lower and higher end
      auto add = [&](int lo, int hi, unsigned mm, double v0, double v1) {
        const double t0 = mm & 1 ? 0.0 : 0.5 * v0, t1 = mm & 2 ? 0.0 : kS3 * v1;
        t[lo] += t0 - t1;
        t[hi] += t0 + t1;
      };
      add(0, 1, m, dd[tri(NT, a, 0) * 64], dd[tri(NT, a, 1) * 64]);
      if (quad) {
        add(2, 3, mu, bo[(a * NT) * 64], bo[(a * NT + 1) * 64]);
        add(0, 2, m >> NT, bo[(2 * NB + a * NT) * 64], bo[(2 * NB + a * NT + 1) * 64]);
        add(1, 3, mr >> NT, bo[(3 * NB + a * NT) * 64], bo[(3 * NB + a * NT + 1) * 64]);
      }
      if (below) {
        add(4, 5, md, bd[a * 64], bd[(NT + a) * 64]);
        add(4, 0, md >> NT, bd[(4 * NB + a * NT) * 64], bd[(4 * NB + a * NT + 1) * 64]);
        add(5, 1, mdr >> NT, bd[(5 * NB + a * NT) * 64], bd[(5 * NB + a * NT + 1) * 64]);
      }
#pragma unroll
      for (int v = 0; v < 6; ++v) out[(v * NT + a) * 64] = (m >> a) & 1 ? 0.0 : t[v];
    }
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      double t[6] = {0, 0, 0, 0, 0, 0};
      auto add = [&](int lo, int hi, unsigned mm, double v0, double v1) {
        const double t0 = mm & 1 ? 0.0 : 0.5 * v0, t1 = mm & 2 ? 0.0 : kS3 * v1;
        t[lo] += t0 - t1;
        t[hi] += t0 + t1;
      };
      add(0, 1, m >> NT, dd[(NS + tri(NT, a, 0)) * 64], dd[(NS + tri(NT, a, 1)) * 64]);
      if (quad) {
        add(2, 3, mr >> NT, bo[(NB + a * NT) * 64], bo[(NB + a * NT + 1) * 64]);
        add(0, 2, m, bo[(2 * NB + a) * 64], bo[(2 * NB + NT + a) * 64]);
        add(1, 3, mu, bo[(4 * NB + a) * 64], bo[(4 * NB + NT + a) * 64]);
      }
      if (left) {
        add(4, 5, ml >> NT, bl[(NB + a) * 64], bl[(NB + NT + a) * 64]);
        add(4, 0, ml, bl[(3 * NB + a) * 64], bl[(3 * NB + NT + a) * 64]);
        add(5, 1, mlu, bl[(5 * NB + a) * 64], bl[(5 * NB + NT + a) * 64]);
      }
#pragma unroll
      for (int v = 0; v < 6; ++v) out[((6 + v) * NT + a) * 64] = (m >> (NT + a)) & 1 ? 0.0 : t[v];
    }
  }
}

// stencils of vertex level 1 from the up to four quads around each vertex
template <class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_l1_kernel(QuadSys S, Sel sel) {
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  // slot of the offset from vertex u to vertex v of a quad (v - u in x, y)
  constexpr int slot[3][3] = {{8, 4, 5}, {2, 0, 1}, {6, 3, 7}};  // [dy + 1][dx + 1]
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.G; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W;
    double st[kStencil];
#pragma unroll
    for (int s = 0; s < kStencil; ++s) st[s] = 0.0;
    const bool fixed = I.vmask[g] != 0;
    if (!fixed) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int qi = i - (u & 1), qj = j - (u >> 1);
        if (qi < 0 || qi >= I.nx || qj < 0 || qj >= I.ny) continue;
        const double* c = S.cq + at<kQuadCq>(I, qj * I.W + qi);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int dx = (v & 1) - (u & 1), dy = (v >> 1) - (u >> 1);
          const int a = u < v ? u : v, b = u < v ? v : u;
          st[slot[dy + 1][dx + 1]] += c[(a * 4 - a * (a - 1) / 2 + b - a) * 64];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < kStencil; ++s) I.l1a[(int64_t)s * I.G + g] = fixed ? (s == 0 ? 1.0 : 0.0) : st[s];
    I.l1dinv[g] = fixed ? 0.0 : 1.0 / st[0];
  }
}

// ------------------------------------------------------------ smoothing weight
__device__ inline double hash01(uint64_t i) {
  uint64_t z = i * 0x9e3779b97f4a7c15ULL + 0x632be59bd9b4e019ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  z ^= z >> 31;
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// y = Dinv_f x for one face (symmetric triangle)
template <int NT, class W>
__device__ __forceinline__ void dinv_apply(const W (&d)[NT * (NT + 1) / 2], const double* x, double* y) {
#pragma unroll
  for (int a = 0; a < NT; ++a) y[a] = 0.0;
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = a; b < NT; ++b) {
      const double v = (double)d[tri(NT, a, b)];
      y[a] = fma(v, x[b], y[a]);
      if (a != b) y[b] = fma(v, x[a], y[b]);
    }
}
template <int NT, class W>
__device__ __forceinline__ void dinv_face(const W* __restrict__ p, const double* x, double* y) {
  W d[NT * (NT + 1) / 2];
#pragma unroll
  for (int s = 0; s < NT * (NT + 1) / 2; ++s) d[s] = p[s * 64];
  dinv_apply<NT>(d, x, y);
}

// RAND: r0 pseudo-random on the free dofs, z = Dinv r0 (Lanczos start);
// otherwise r0 = the reduced load, x = 0.  p = q = 0.  (b, b) is that of the
// whole trace system, diagonals included.
template <int NT, bool RAND, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_init_kernel(QuadSys S, Sel sel) {
  constexpr int NV = 2 * NT, NS = NT * (NT + 1) / 2, NC = 4 * NT;
  __shared__ double sh[kNW];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  double prz = 0.0, pbb = 0.0;
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.ntiles * 64; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W;
    const unsigned m = S.mask[(I.tile0 << 6) + g];
    const int64_t o = at<NV>(I, g);
    const bool in = g < I.G, quad = in && i < I.nx && j < I.ny;
    const bool below = in && j > 0 && i < I.nx, left = in && i > 0 && j < I.ny;
    double r[NV];
    if constexpr (RAND) {
#pragma unroll
      for (int a = 0; a < NV; ++a) r[a] = (m >> a) & 1 ? 0.0 : hash01((uint64_t)g * NV + a) - 0.5;
    } else {
      const double* bo = S.bq + at<9 * NT>(I, g);
      const double* bd = S.bq + at<9 * NT>(I, below ? g - I.W : g);
      const double* bl = S.bq + at<9 * NT>(I, left ? g - 1 : g);
#pragma unroll
      for (int a = 0; a < NV; ++a) {
        // H: B of the quad, T of the one below; V: L, and R of the one to the left
        const int f = a / NT, c = (2 * f) * NT + a - f * NT, c2 = c + NT;
        const double* n = f ? bl : bd;
        const bool other = f ? left : below;
        double red = (quad ? bo[c * 64] : 0.0) + (other ? n[c2 * 64] : 0.0);
        const double raw = (quad ? bo[(NC + c) * 64] : 0.0) + (other ? n[(NC + c2) * 64] : 0.0);
        if ((m >> a) & 1) red = 0.0;
        else pbb = fma(raw, raw, pbb);
        r[a] = red;
      }
      if (quad)
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          const double d = bo[(2 * NC + a) * 64];
          pbb = fma(d, d, pbb);
        }
    }
#pragma unroll
    for (int a = 0; a < NV; ++a) {
      S.r0[o + a * 64] = r[a];
      S.p[o + a * 64] = 0.0;
      S.q[o + a * 64] = 0.0;
      if (!RAND) S.x[o + a * 64] = 0.0;
    }
    if constexpr (RAND) {
      if (in) {
        const double* d = S.Dinv + at<2 * NS>(I, g);
        double y[NV];
        dinv_face<NT>(d, r, y);
        dinv_face<NT>(d + NS * 64, r + NT, y + NT);
#pragma unroll
        for (int a = 0; a < NV; ++a) {
          S.z[o + a * 64] = y[a];
          prz = fma(r[a], y[a], prz);
        }
      }
    }
  }
  if (RAND) {
    const double s = bsum(prz, sh);
    if (threadIdx.x == 0) S.part[(size_t)S.nbt + I.pE + lb] = s;
  } else {
    const double s = bsum(pbb, sh);
    if (threadIdx.x == 0) S.part[(size_t)S.nbt * 4 + I.pE + lb] = s;
  }
  if (lb == 0 && threadIdx.x == 0) {
    I.st->done = 0;
    I.st->it = 0;
    I.st->pq = 0.0;
    I.st->i_pre = 0;
    I.st->i_upd = 0;
    I.st->i_spmv = 1;
  }
}

// block-Jacobi update of the Lanczos run: r -= alpha q, z = Dinv r
template <int NT, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_lupd_kernel(QuadSys S, Sel sel) {
  constexpr int NV = 2 * NT, NS = NT * (NT + 1) / 2;
  __shared__ double sh[kNW];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  CgState* st = I.st;
  const int done = st->done, it = st->i_upd;
  const double rz2[2] = {st->rz[0], st->rz[1]};
  const double ps = pshare(S.part + I.pM, I.nbM);
  if (done) return;
  if (lb == 0 && threadIdx.x == 0) st->i_spmv = it + 1;
  const double pq = bsum(ps, sh);
  if (!(pq > 0.0)) {
    if (lb == 0 && threadIdx.x == 0) {
      st->done = 3;
      st->it = it - 1;
    }
    return;
  }
  if (lb == 0 && threadIdx.x == 0) st->lpq[it] = pq;
  const double alpha = (it & 1 ? rz2[1] : rz2[0]) / pq;
  double prz = 0.0;
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.G; g += I.nbE * kQuadThreads) {
    const int64_t o = at<NV>(I, g);
    const double* d = S.Dinv + at<2 * NS>(I, g);
    double r[NV], y[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) {
      r[a] = fma(-alpha, S.q[o + a * 64], S.r0[o + a * 64]);
      S.r0[o + a * 64] = r[a];
    }
    dinv_face<NT>(d, r, y);
    dinv_face<NT>(d + NS * 64, r + NT, y + NT);
#pragma unroll
    for (int a = 0; a < NV; ++a) {
      S.z[o + a * 64] = y[a];
      prz = fma(r[a], y[a], prz);
    }
  }
  const double s = bsum(prz, sh);
  if (threadIdx.x == 0) S.part[(size_t)S.nbt + I.pE + lb] = s;
}

// omega = factor / (largest eigenvalue of the Lanczos tridiagonal matrix of
// the m completed steps), by bisection on Sturm counts to 1e-4 (the weight
// is not sensitive to more); 0.5 when no step completed.  One block per
// instance; the last step's (p, q) is summed here.
template <class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_omega_kernel(QuadSys S, Sel sel, int m, double factor) {
  __shared__ double sh[kNW];
  const QuadInst& I = inst_block(sel);
  CgState* st = I.st;
  const int done = st->done, its = st->it;
  double lz[kLanczos + 2], lpq[kLanczos + 1];
#pragma unroll
  for (int j = 1; j <= kLanczos; ++j) {
    lz[j] = st->lz[j];
    lpq[j] = st->lpq[j];
  }
  lz[kLanczos + 1] = 0.0;
  const double pq = bsum(pshare(S.part + I.pM, I.nbM), sh);
  if (threadIdx.x != 0) return;
  if (done) {
    m = min(m, its);
  } else {
    st->lpq[m] = pq;
#pragma unroll
    for (int j = 1; j <= kLanczos; ++j) lpq[j] = j == m ? pq : lpq[j];
  }
  double d[kLanczos], e2[kLanczos];
  int n = 0;
#pragma unroll
  for (int j = 1; j <= kLanczos; ++j) {
    if (j > m || n != j - 1) continue;
    const double a = lz[j] / lpq[j];
    double dj = 1.0 / a;
    if (j > 1) dj += (lz[j] / lz[j - 1]) / (lz[j - 1] / lpq[j - 1]);
    if (!(dj > 0.0) || !isfinite(dj)) continue;
    d[j - 1] = dj;
    e2[j - 1] = j < m ? (lz[j + 1] / lz[j]) / (a * a) : 0.0;
    if (!isfinite(e2[j - 1])) continue;
    n = j;
  }
  if (n == 0) {
    st->omega = 0.5;
    return;
  }
  double hi = 0.0;
  for (int j = 0; j < n; ++j) {
    const double r = (j > 0 ? sqrt(e2[j - 1]) : 0.0) + (j + 1 < n ? sqrt(e2[j]) : 0.0);
    hi = fmax(hi, d[j] + r);
  }
  double lo = 0.0;
  while (hi - lo > 1e-4 * hi) {
    const double x = 0.5 * (lo + hi);
    int below = 0;
    double q = 1.0;
    for (int j = 0; j < n; ++j) {
      q = d[j] - x - (j > 0 ? e2[j - 1] / q : 0.0);
      if (q == 0.0) q = -1e-300;
      below += q < 0.0;
    }
    if (below < n) lo = x;
    else hi = x;
  }
  st->omega = factor / hi;
}

// --------------------------------------------------------------- CG kernels
// The couplings of quad (i, j) applied to the four faces' values, rows added
// to y.  A face's row block uses the neighbours' mode 0 less its own shift
// s (0, or its own mode 0 where the system annihilates constants: the row
// then acts on differences, and the rounding of the stored entries no longer
// feeds the smooth part of the solution).
template <int NT, class V>
__device__ __forceinline__ void pair_apply(const V (&v)[NT * NT], const double* X, const double* Y, double sx,
                                           double sy, double* yX, double* yY) {
  const double x0 = X[0] - sy, y0 = Y[0] - sx;
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      const double w = (double)v[a * NT + b];
      yX[a] = fma(w, b == 0 ? y0 : Y[b], yX[a]);
      yY[b] = fma(w, a == 0 ? x0 : X[a], yY[b]);
    }
}
template <int N, class V>
__device__ __forceinline__ void load_vals(const V* __restrict__ p, V (&b)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) b[k] = __builtin_nontemporal_load(p + k * 64);
}
// The walks load a row's couplings one block ahead of their use: what is
// loaded through p after after<NT>(p, x, y) waits for the sums x and y to be
// formed.  Left to itself the compiler loads all six blocks at once, which
// spills at 4 and 5 modes (1024^2 P3: residual 646 us), or each at its use
// (561 us).
template <int NT, class V>
__device__ __forceinline__ void after(const V*& p, double* x, double* y) {
#pragma unroll
  for (int a = 0; a < NT; ++a) {
    asm volatile("" : "+v"(x[a]));
    asm volatile("" : "+v"(y[a]));
  }
  asm volatile("" : "+v"(p));
}

__device__ __forceinline__ double shift_up(double v) { return __shfl_up(v, 1, 64); }
__device__ __forceinline__ double shift_down(double v) { return __shfl_down(v, 1, 64); }

// CG product.  A wavefront walks R grid rows upwards over 62 columns (lane 0
// repeats the column to the left for its contribution to the first V, lane 63
// only lends its V): each quad's couplings are loaded once and serve its four
// faces, the contribution to T carried to the next row in registers and that
// to R handed to the next lane.  Row groups are laid end to end, so a
// wavefront may run over the end of one group into the next.  HBM-bound:
// 6 nt^2 + nt (nt+1) values of the matrix, 6 nt in and 4 nt out per point.
// A window's 63 columns touch 4.9 cache lines on average where 62 doubles fill
// 3.9; the rest is the next window's, so consecutive windows run on one XCD
// (xcd_task).
template <int NT, bool LANCZOS, class Sel>
__global__ __launch_bounds__(kQuadThreads, NT == 2 ? 4 : (NT == 3 ? 3 : 2)) void q_product_kernel(QuadSys S, Sel sel, double rtol2, int maxit,
                                                                   int force) {
  constexpr int NV = 2 * NT, NB = NT * NT, NS = NT * (NT + 1) / 2;
  __shared__ double sh[kNW];
  __shared__ double cs[(kNW + 1) * NT * 64];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  lb = xcd_task(lb, I.nbM);
  CgState* st = I.st;
  const size_t nbt = (size_t)S.nbt;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ncol = I.W * I.NG;
  const int done = st->done, it = force ? 2 : st->i_spmv, plain = *I.plain;
  const double rz2[2] = {st->rz[0], st->rz[1]};
  // z of the row a task starts on, loaded ahead of it
  double zB[NT];
  const auto start_row = [&](int task) {
    const int c = task * kQuadOwn - 1 + lane;
    const bool valid = c >= 0 && c < ncol;
    const int grp = valid ? c / I.W : 0, i = valid ? c - grp * I.W : 0;
    const int j = (grp * kNW + wave) * I.R + (wave == 0 ? -1 : 0);
    const double* zp = S.z + at<NV>(I, valid && j >= 0 && j <= I.ny ? j * I.W + i : I.nx);
#pragma unroll
    for (int a = 0; a < NT; ++a) zB[a] = zp[a * 64];
  };
  start_row(lb);
  const double ps = pshare(S.part + nbt + I.pE, I.nbE);
  if (!force && done) return;
  const double rz = bsum(ps, sh);
  const bool lead = lb == 0 && threadIdx.x == 0;
  if constexpr (LANCZOS) {
    if (!(rz > 0.0)) {
      if (lead) {
        st->done = 1;
        st->it = it - 1;
      }
      return;
    }
    if (lead) {
      st->rz[it & 1] = rz;
      st->it = it - 1;
      st->i_upd = it;
      st->lz[it] = rz;
    }
  } else if (!force) {
    // the first vertex kernel takes the convergence test after every update;
    // the initial residual is tested here
    if (it == 1) {
      const double rr = psum(S.part + nbt * 3 + I.pM, I.nbM, sh);
      const double bb = psum(S.part + nbt * 4 + I.pE, I.nbE, sh);
      const bool conv = rr <= rtol2 * bb;
      if (lead) {
        st->it = 0;
        st->rr = rr;
        st->bb = bb;
        if (conv || maxit < 1) st->done = conv ? 1 : 2;
      }
      if (conv || maxit < 1) return;
    }
    if (lead) {
      st->rz[it & 1] = rz;
      st->i_upd = it;
    }
  }
  const double beta = it == 1 ? 0.0 : (force ? 0.5 : rz / (it & 1 ? rz2[0] : rz2[1]));
  const double sf = S.shift && !plain ? 1.0 : 0.0;
  double part = 0.0;
  for (int task = lb; task < I.tasks; task += I.nbM) {
    const int c = task * kQuadOwn - 1 + lane;
    const bool valid = c >= 0 && c < ncol;
    const int grp = valid ? c / I.W : 0, i = valid ? c - grp * I.W : 0, j0 = (grp * kNW + wave) * I.R;
    const bool own = valid && lane >= 1 && lane < 63;
    const int first = wave == 0 ? -1 : 0;
    double carry[NT], y0[NT];
#pragma unroll
    for (int a = 0; a < NT; ++a) carry[a] = y0[a] = 0.0;
    if (task != lb) start_row(task);
    for (int s = first; s < I.R; ++s) {
      const int j = j0 + s;
      const bool ok = valid && j >= 0 && j <= I.ny, up = valid && j + 1 <= I.ny;
      const int g = ok ? j * I.W + i : I.nx;
      const double* zp = S.z + at<NV>(I, g) + NT * 64;
      const double* zu = S.z + at<NV>(I, up ? (j + 1) * I.W + i : I.nx);
      const double* v = S.blk + at<6 * NB>(I, lane < 63 ? g : I.nx);
      double zT[NT], zL[NT], zR[NT], b0[NB], b1[NB];
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const double t = zp[a * 64];
        zL[a] = ok ? t : 0.0;
        zT[a] = zu[a * 64];
      }
      load_vals(v, b0);
      load_vals(v + 4 * NB * 64, b1);
#pragma unroll
      for (int a = 0; a < NT; ++a) zR[a] = shift_down(zL[a]);
      double yB[NT], yT[NT], yL[NT], yR[NT];
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        yB[a] = carry[a];
        yT[a] = yL[a] = yR[a] = 0.0;
      }
      const double sB = sf * zB[0], sT = sf * zT[0], sL = sf * zL[0], sR = sf * zR[0];
      pair_apply<NT>(b0, zB, zT, sB, sT, yB, yT);
      after<NT>(v, yB, yT);
      load_vals(v + 5 * NB * 64, b0);
      pair_apply<NT>(b1, zT, zL, sT, sL, yT, yL);
      if (s < 0) {
        pair_apply<NT>(b0, zT, zR, sT, sR, yT, yR);
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          cs[(0 * NT + a) * 64 + lane] = yT[a];
          carry[a] = 0.0;
          zB[a] = zT[a];
        }
        continue;
      }
      after<NT>(v, yT, yL);
      load_vals(v + NB * 64, b1);
      pair_apply<NT>(b0, zT, zR, sT, sR, yT, yR);
      after<NT>(v, yT, yR);
      load_vals(v + 2 * NB * 64, b0);
      pair_apply<NT>(b1, zL, zR, sL, sR, yL, yR);
      after<NT>(v, yL, yR);
      load_vals(v + 3 * NB * 64, b1);
      const unsigned m = S.mask[(I.tile0 << 6) + g];
      const int64_t o = at<NV>(I, g);
      const double* dp = S.D + at<2 * NS>(I, g);
      const double *qp = S.q + o, *pp = S.p + o;
      double d[2 * NS], qo[NV], po[NV];
      pair_apply<NT>(b0, zB, zL, sB, sL, yB, yL);
      after<NT>(dp, yB, yL);
      load_vals(dp, d);
      pair_apply<NT>(b1, zB, zR, sB, sR, yB, yR);
      after<NT>(qp, yB, yR);
      after<NT>(pp, yB, yR);
#pragma unroll
      for (int a = 0; a < NV; ++a) {
        qo[a] = qp[a * 64];
        po[a] = pp[a * 64];
      }
      const double h0 = zB[0] - sB, l0 = zL[0] - sL;
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = a; b < NT; ++b) {
          const double h = d[tri(NT, a, b)], w = d[NS + tri(NT, a, b)];
          yB[a] = fma(h, b == 0 ? h0 : zB[b], yB[a]);
          yL[a] = fma(w, b == 0 ? l0 : zL[b], yL[a]);
          if (a != b) {
            yB[b] = fma(h, a == 0 ? h0 : zB[a], yB[b]);
            yL[b] = fma(w, a == 0 ? l0 : zL[a], yL[b]);
          }
        }
#pragma unroll
      for (int a = 0; a < NT; ++a) yL[a] += shift_up(yR[a]);
      if (own && ok) {
#pragma unroll
        for (int a = 0; a < NV; ++a) {
          if (a < NT && s == 0) continue;
          const double y = (m >> a) & 1 ? 0.0 : (a < NT ? yB[a] : yL[a - NT]);
          const double zv = a < NT ? zB[a] : zL[a - NT];
          const double qn = fma(beta, qo[a], y), pn = fma(beta, po[a], zv);
          S.q[o + a * 64] = qn;
          S.p[o + a * 64] = pn;
          part = fma(pn, qn, part);
        }
      }
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        if (s == 0) y0[a] = yB[a];
        carry[a] = yT[a];
        zB[a] = zT[a];
      }
    }
    // the first row's H, with the contribution of the row below it
    const bool ok = valid && j0 <= I.ny;
    const int g = ok ? j0 * I.W + i : I.nx;
    const int64_t o = at<NV>(I, g);
    const unsigned m = S.mask[(I.tile0 << 6) + g];
    double qo[NT], po[NT], zv[NT];
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      cs[((wave + 1) * NT + a) * 64 + lane] = carry[a];
      qo[a] = S.q[o + a * 64];
      po[a] = S.p[o + a * 64];
      zv[a] = S.z[o + a * 64];
    }
    __syncthreads();
    if (own && ok) {
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const double y = (m >> a) & 1 ? 0.0 : y0[a] + cs[(wave * NT + a) * 64 + lane];
        const double qn = fma(beta, qo[a], y), pn = fma(beta, po[a], zv[a]);
        S.q[o + a * 64] = qn;
        S.p[o + a * 64] = pn;
        part = fma(pn, qn, part);
      }
    }
    __syncthreads();
  }
  const double t = bsum(part, sh);
  if (threadIdx.x == 0) S.part[I.pM + lb] = t;
}

// Update and level-0 residual: r' = r - alpha q, e0 = omega Dinv r' formed at
// every face the quads touch, res = r' - T e0 (T_ff e0_f = omega r' on free
// rows, so the diagonal blocks are not read), and the restriction of res to
// the vertices, by the product's walk.  The row below the group is walked in
// full for the restriction's lower neighbour.  Matrix and Dinv stored as W.
template <int NT, class W, class Sel>
__global__ __launch_bounds__(kQuadThreads, NT == 2 ? 4 : (NT == 3 ? 3 : 2)) void q_residual_kernel(QuadSys S, Sel sel, const W* __restrict__ blk,
                                                                    const W* __restrict__ Dinv, int force) {
  constexpr int NV = 2 * NT, NB = NT * NT, NS = NT * (NT + 1) / 2;
  __shared__ double sh[kNW];
  __shared__ double cs[(kNW + 1) * NT * 64], hs[(kNW + 1) * 64];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  lb = xcd_task(lb, I.nbM);
  CgState* st = I.st;
  // the initial residual (0, nothing to update) or iteration i_upd
  const int done = st->done, it = force ? 2 : st->i_upd;
  const double rz2[2] = {st->rz[0], st->rz[1]}, om = st->omega;
  const size_t nbt = (size_t)S.nbt;
  const double ps = pshare(S.part + I.pM, I.nbM);
  if (!force && done) return;
  double alpha = 0.0;
  if (!force) {
    if (it > 0) {
      const double pq = bsum(ps, sh);
      if (!(pq > 0.0)) {
        if (lb == 0 && threadIdx.x == 0) {
          st->done = 3;
          st->it = it - 1;
        }
        return;
      }
      alpha = (it & 1 ? rz2[1] : rz2[0]) / pq;
    }
    if (lb == 0 && threadIdx.x == 0) st->i_pre = it;
  }
  const double* __restrict__ rin = it & 1 ? S.r1 : S.r0;
  double* __restrict__ rout = it & 1 ? S.r0 : S.r1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ncol = I.W * I.NG;
  double prr = 0.0;
  for (int task = lb; task < I.tasks; task += I.nbM) {
    const int c = task * kQuadOwn - 1 + lane;
    const bool valid = c >= 0 && c < ncol;
    const int grp = valid ? c / I.W : 0, i = valid ? c - grp * I.W : 0, j0 = (grp * kNW + wave) * I.R;
    const bool own = valid && lane >= 1 && lane < 63;
    const int first = wave == 0 ? -1 : 0;
    double carry[NT], eB[NT], rB[NT], y0[NT], r0[NT], hiV = 0.0, loV0 = 0.0;
    {
      const int j = j0 + first;
      const int g = valid && j >= 0 && j <= I.ny ? j * I.W + i : I.nx;
      const int64_t o = at<NV>(I, g);
#pragma unroll
      for (int a = 0; a < NT; ++a) rB[a] = fma(-alpha, S.q[o + a * 64], rin[o + a * 64]);
      dinv_face<NT>(Dinv + at<2 * NS>(I, g), rB, eB);
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        eB[a] *= om;
        carry[a] = y0[a] = r0[a] = 0.0;
      }
    }
    for (int s = first; s < I.R; ++s) {
      const int j = j0 + s;
      const bool ok = valid && j >= 0 && j <= I.ny;
      const int g = ok ? j * I.W + i : I.nx;
      const int64_t o = at<NV>(I, g);
      const W* v = blk + at<6 * NB>(I, lane < 63 ? g : I.nx);
      double rT[NT], eT[NT], rL[NT], eL[NT], eR[NT];
      W b0[NB], b1[NB], dT[NS], dL[NS];
      const int gT = valid && j + 1 <= I.ny ? (j + 1) * I.W + i : I.nx;
      const int64_t oT = at<NV>(I, gT);
      load_vals(Dinv + at<2 * NS>(I, gT), dT);
      load_vals(Dinv + at<2 * NS>(I, g) + NS * 64, dL);
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        rT[a] = fma(-alpha, S.q[oT + a * 64], rin[oT + a * 64]);
        const double t = fma(-alpha, S.q[o + (NT + a) * 64], rin[o + (NT + a) * 64]);
        rL[a] = ok ? t : 0.0;
      }
      load_vals(v, b0);
      load_vals(v + 4 * NB * 64, b1);
      dinv_apply<NT>(dT, rT, eT);
      dinv_apply<NT>(dL, rL, eL);
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        eT[a] *= om;
        eL[a] *= om;
        eR[a] = shift_down(eL[a]);
      }
      double yB[NT], yT[NT], yL[NT], yR[NT];
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        yB[a] = carry[a];
        yT[a] = yL[a] = yR[a] = 0.0;
      }
      pair_apply<NT>(b0, eB, eT, 0.0, 0.0, yB, yT);
      after<NT>(v, yB, yT);
      load_vals(v + 5 * NB * 64, b0);
      pair_apply<NT>(b1, eT, eL, 0.0, 0.0, yT, yL);
      after<NT>(v, yT, yL);
      load_vals(v + NB * 64, b1);
      pair_apply<NT>(b0, eT, eR, 0.0, 0.0, yT, yR);
      after<NT>(v, yT, yR);
      load_vals(v + 2 * NB * 64, b0);
      pair_apply<NT>(b1, eL, eR, 0.0, 0.0, yL, yR);
      after<NT>(v, yL, yR);
      load_vals(v + 3 * NB * 64, b1);
      const double *xp = S.x + o, *pp = S.p + o;
      const unsigned mk = S.mask[(I.tile0 << 6) + g];
      const unsigned char vm = I.vmask[g];
      double xo[NV], po[NV];
      pair_apply<NT>(b0, eB, eL, 0.0, 0.0, yB, yL);
      after<NT>(xp, yB, yL);
      after<NT>(pp, yB, yL);
#pragma unroll
      for (int a = 0; a < NV; ++a) {
        xo[a] = xp[a * 64];
        po[a] = pp[a * 64];
      }
      pair_apply<NT>(b1, eB, eR, 0.0, 0.0, yB, yR);
#pragma unroll
      for (int a = 0; a < NT; ++a) yL[a] += shift_up(yR[a]);
      const unsigned m = ok ? mk : ~0u;
      double sB[NT], sL[NT];
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        sB[a] = (m >> a) & 1 ? 0.0 : fma(-om, rB[a], rB[a]) - yB[a];
        sL[a] = (m >> (NT + a)) & 1 ? 0.0 : fma(-om, rL[a], rL[a]) - yL[a];
      }
      // P^T res: H from its lower end (this vertex) and its higher end (the
      // next lane's), V from its lower end and, one row up, its higher end
      const double loH = fma(-kS3, sB[1], 0.5 * sB[0]), hiH = fma(kS3, sB[1], 0.5 * sB[0]);
      const double loV = fma(-kS3, sL[1], 0.5 * sL[0]);
      const double hiL = shift_up(hiH);
      if (s >= 0 && own && ok) {
        if (s > 0) I.r1[g] = vm ? 0.0 : ((loH + loV) + hiL) + hiV;
#pragma unroll
        for (int a = 0; a < NV; ++a) {
          if (a < NT && s == 0) continue;
          const double rn = a < NT ? rB[a] : rL[a - NT];
          S.res[o + a * 64] = a < NT ? sB[a] : sL[a - NT];
          rout[o + a * 64] = rn;
          prr = fma(rn, rn, prr);
          S.x[o + a * 64] = fma(alpha, po[a], xo[a]);
        }
      }
      hiV = fma(kS3, sL[1], 0.5 * sL[0]);
      if (s < 0) {
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          cs[a * 64 + lane] = yT[a];
          yT[a] = 0.0;
        }
        hs[lane] = hiV;
      } else if (s == 0) {
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          y0[a] = yB[a];
          r0[a] = rB[a];
        }
        loV0 = loV;
      }
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        carry[a] = yT[a];
        eB[a] = eT[a];
        rB[a] = rT[a];
      }
    }
    // the first row's H and its vertices, with what the row below adds
    const bool ok = valid && j0 <= I.ny;
    const int g = ok ? j0 * I.W + i : I.nx;
    const int64_t o = at<NV>(I, g);
    const unsigned m = ok ? S.mask[(I.tile0 << 6) + g] : ~0u;
    const unsigned char vm = I.vmask[g];
    double xo[NT], po[NT], sB[NT];
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      cs[((wave + 1) * NT + a) * 64 + lane] = carry[a];
      xo[a] = S.x[o + a * 64];
      po[a] = S.p[o + a * 64];
    }
    hs[(wave + 1) * 64 + lane] = hiV;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NT; ++a)
      sB[a] = (m >> a) & 1 ? 0.0 : fma(-om, r0[a], r0[a]) - (y0[a] + cs[(wave * NT + a) * 64 + lane]);
    const double loH = fma(-kS3, sB[1], 0.5 * sB[0]), hiH = fma(kS3, sB[1], 0.5 * sB[0]);
    const double hiL = shift_up(hiH);
    if (own && ok) {
      I.r1[g] = vm ? 0.0 : ((loH + loV0) + hiL) + hs[wave * 64 + lane];
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        S.res[o + a * 64] = sB[a];
        rout[o + a * 64] = r0[a];
        prr = fma(r0[a], r0[a], prr);
        S.x[o + a * 64] = fma(alpha, po[a], xo[a]);
      }
    }
    __syncthreads();
  }
  const double t = bsum(prr, sh);
  if (threadIdx.x == 0) S.part[nbt * 3 + I.pM + lb] = t;
}

// z = P e1 + omega Dinv (r + res - (T P) e1), pointwise (hdg_quad.h)
template <int NT, class W, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_smooth_kernel(QuadSys S, Sel sel, const W* __restrict__ tp,
                                                               const W* __restrict__ Dinv) {
  constexpr int NV = 2 * NT, NS = NT * (NT + 1) / 2;
  __shared__ double sh[kNW];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  CgState* st = I.st;
  const int done = st->done, it = st->i_pre;
  const double om = st->omega;
  if (done) return;
  if (lb == 0 && threadIdx.x == 0) st->i_spmv = it + 1;
  const double* __restrict__ r = it & 1 ? S.r0 : S.r1;
  const double* __restrict__ e1 = I.e1;
  double prz = 0.0;
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.G; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W, W_ = I.W;
    const unsigned m = S.mask[(I.tile0 << 6) + g];
    const int64_t o = at<NV>(I, g);
    const W* t = tp + at<12 * NT>(I, g);
    const W* d = Dinv + at<2 * NS>(I, g);
    const bool xr = i < I.nx, yu = j < I.ny, xl = i > 0, yd = j > 0;
    const double e00 = e1[g], e10 = xr ? e1[g + 1] : 0.0, e01 = yu ? e1[g + W_] : 0.0;
    const double e11 = xr && yu ? e1[g + W_ + 1] : 0.0;
    const double ed0 = yd ? e1[g - W_] : 0.0, ed1 = yd && xr ? e1[g - W_ + 1] : 0.0;
    const double el0 = xl ? e1[g - 1] : 0.0, el1 = xl && yu ? e1[g - 1 + W_] : 0.0;
    const double eh[6] = {e00, e10, e01, e11, ed0, ed1}, ev[6] = {e00, e01, e10, e11, el0, el1};
    double rv[NV], s[NV], y[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) {
      rv[a] = r[o + a * 64];
      s[a] = rv[a] + S.res[o + a * 64];
    }
#pragma unroll
    for (int v = 0; v < 6; ++v)
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        s[a] = fma(-(double)__builtin_nontemporal_load(t + (v * NT + a) * 64), eh[v], s[a]);
        s[NT + a] = fma(-(double)__builtin_nontemporal_load(t + ((6 + v) * NT + a) * 64), ev[v], s[NT + a]);
      }
    dinv_face<NT>(d, s, y);
    dinv_face<NT>(d + NS * 64, s + NT, y + NT);
    const double ph0 = 0.5 * (e00 + e10), ph1 = kS3 * (e10 - e00), pv0 = 0.5 * (e00 + e01), pv1 = kS3 * (e01 - e00);
#pragma unroll
    for (int a = 0; a < NV; ++a) {
      const double pe = a == 0 ? ph0 : (a == 1 ? ph1 : (a == NT ? pv0 : (a == NT + 1 ? pv1 : 0.0)));
      const double zv = (m >> a) & 1 ? 0.0 : fma(om, y[a], pe);
      S.z[o + a * 64] = zv;
      prz = fma(rv[a], zv, prz);
    }
  }
  const double b = bsum(prz, sh);
  if (threadIdx.x == 0) S.part[(size_t)S.nbt + I.pE + lb] = b;
}

// ----------------------------------------------------------------- finish
// uhat in the natural numbering: the axis faces' x (prescribed values on
// their dofs), and the diagonals from their own rows,
// K_DD x_D = rhs_D - K_Do uhat_o.  With `resid`, the quads' parts of K uhat -
// rhs on their five faces go to bq (slots B T L R, then D).
template <int NT, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_finish_kernel(QuadSys S, Sel sel, double* __restrict__ uhat,
                                                               int resid) {
  constexpr int NTR = 3 * NT, CA = NTR * NTR, LPQ = lanes_per_quad(NT), QB = quads_per_block(NT);
  constexpr int NV = 2 * NT, NC = 4 * NT;
  constexpr int QS = quad_stride(NT);
  __shared__ double A[QB * QS];
  __shared__ double bs[QB * 2 * NTR], us[QB * 2 * NTR];
  __shared__ double ts[QB * NT];
  __shared__ unsigned char ms[QB * NT];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  const int nquads = I.nx * I.ny;
  const int q0 = lb * QB, nq = min(QB, nquads - q0);
  CellFetch<NT> cells;
  if (!S.from_k) cells.fetch(S, I, q0, nq);
  if (S.from_k)
    stage_assembled<NT>(S, I, q0, nq, A, bs);
  else
    cells.stage(A, bs, nq);
  // the cells' trace values (D: the prescribed ones, zero on its free dofs)
  for (int e = threadIdx.x; e < nq * 2 * NTR; e += kQuadThreads) {
    const int ql = e / (2 * NTR), cell = (e / NTR) & 1, r = e % NTR, lr = r / NT, a = r % NT;
    const int q = q0 + ql, i = q % I.nx, j = q / I.nx;
    const int64_t f = S.cf[3 * (I.cell0 + 2 * (int64_t)q + cell) + lr];
    const bool dm = S.dmask[f * NT + a] != 0;
    double u = dm ? S.uD[f * NT + a] : 0.0;
    if (lr == cell) {
      if (cell == 0) ms[ql * NT + a] = dm;
    } else if (!dm) {
      // lower: L (1), B (2); upper: T (0), R (2)
      const int g = j * I.W + i;
      const bool isv = cell == 0 ? lr == 1 : lr == 2;
      const int gp = cell == 0 ? g : (lr == 0 ? g + I.W : g + 1);
      u = S.x[at<NV>(I, gp) + (isv ? NT + a : a) * 64];
    }
    us[e] = u;
    // each axis face is written by the quad it is B or L of, or by the last
    // quad of its column or row
    if (lr != cell && (cell == 0 || (lr == 0 ? j == I.ny - 1 : i == I.nx - 1))) uhat[f * NT + a] = u;
  }
  __syncthreads();
  const int ql = threadIdx.x / LPQ, c = threadIdx.x % LPQ;
  const bool live = ql < nq;
  const double* Al = A + ql * QS;
  const double* Au = Al + CA;
  const double* ul = us + ql * 2 * NTR;
  const double* bl = bs + ql * 2 * NTR;
  if (live && c < NT) {
    double t = bl[c] + bl[NTR + NT + c];
    for (int k = 0; k < NTR; ++k) t = fma(-Al[c * NTR + k], ul[k], t);
    for (int k = 0; k < NTR; ++k) t = fma(-Au[(NT + c) * NTR + k], ul[NTR + k], t);
    ts[ql * NT + c] = t;
  }
  __syncthreads();
  if (live && c == 0) {
    const unsigned char* mD = ms + ql * NT;
    auto masked = [&](int a) { return mD[a] != 0; };
    const DiagFactor<NT> F = factor_d<NT>(Al, Au, masked);
    double y[NT];
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      double t = masked(a) ? 0.0 : -ts[ql * NT + a];
#pragma unroll
      for (int k = 0; k < a; ++k) t = fma(-F.l[a][k], y[k], t);
      y[a] = t;
    }
#pragma unroll
    for (int a = NT - 1; a >= 0; --a) {
      double t = y[a] * F.di[a];
#pragma unroll
      for (int k = a + 1; k < NT; ++k) t = fma(-F.l[k][a], y[k], t);
      y[a] = t;
    }
    const int64_t f = S.cf[3 * (I.cell0 + 2 * (int64_t)(q0 + ql))];
    double* uw = us + ql * 2 * NTR;
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      const double v = masked(a) ? uw[a] : y[a];
      uhat[f * NT + a] = v;
      uw[a] = v;
      uw[NTR + NT + a] = v;
    }
  }
  __syncthreads();
  if (resid && live && c < NC) {
    const int q = q0 + ql, g = (q / I.nx) * I.W + q % I.nx;
    double* out = S.bq + at<9 * NT>(I, g);
    {
      const int f = c / NT, b = c - f * NT, cell = f & 1, lf = f == 0 ? 2 : (f == 1 ? 0 : (f == 2 ? 1 : 2));
      const double* row = (cell ? Au : Al) + (lf * NT + b) * NTR;
      double t = -bl[cell * NTR + lf * NT + b];
      for (int k = 0; k < NTR; ++k) t = fma(row[k], ul[cell * NTR + k], t);
      out[c * 64] = t;
    }
    if (c < NT) {
      double t = -(bl[c] + bl[NTR + NT + c]);
      for (int k = 0; k < NTR; ++k) t = fma(Al[c * NTR + k], ul[k], t);
      for (int k = 0; k < NTR; ++k) t = fma(Au[(NT + c) * NTR + k], ul[NTR + k], t);
      out[(2 * NC + c) * 64] = ms[ql * NT + c] ? 0.0 : t;
    }
  }
}

// per-block partials of ||K uhat - rhs||^2 from the quads' parts
template <int NT, class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_resnorm_kernel(QuadSys S, Sel sel) {
  constexpr int NV = 2 * NT, NC = 4 * NT;
  __shared__ double sh[kNW];
  int lb;
  const QuadInst& I = inst_of(sel, lb);
  double acc = 0.0;
  for (int g = lb * kQuadThreads + threadIdx.x; g < I.G; g += I.nbE * kQuadThreads) {
    const int i = g % I.W, j = g / I.W;
    const unsigned m = S.mask[(I.tile0 << 6) + g];
    const bool quad = i < I.nx && j < I.ny, below = j > 0 && i < I.nx, left = i > 0 && j < I.ny;
    const double* bo = S.bq + at<9 * NT>(I, g);
    const double* bd = S.bq + at<9 * NT>(I, below ? g - I.W : g);
    const double* bl = S.bq + at<9 * NT>(I, left ? g - 1 : g);
#pragma unroll
    for (int a = 0; a < NV; ++a) {
      const int f = a / NT, c = (2 * f) * NT + a - f * NT;
      const double t = (quad ? bo[c * 64] : 0.0) + ((f ? left : below) ? (f ? bl : bd)[(c + NT) * 64] : 0.0);
      if (!((m >> a) & 1)) acc = fma(t, t, acc);
    }
    if (quad)
#pragma unroll
      for (int a = 0; a < NT; ++a) acc = fma(bo[(2 * NC + a) * 64], bo[(2 * NC + a) * 64], acc);
  }
  const double b = bsum(acc, sh);
  if (threadIdx.x == 0) S.part[I.pE + lb] = b;
}

template <class Sel>
__global__ __launch_bounds__(kQuadThreads) void q_sum_kernel(QuadSys S, Sel sel, double* out) {
  __shared__ double sh[kNW];
  const QuadInst& I = inst_block(sel);
  const double s = psum(S.part + I.pE, I.nbE, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

#define Q_NT(nt, CALL)          \
  switch (nt) {                 \
    case 2: CALL(2); break;     \
    case 3: CALL(3); break;     \
    case 4: CALL(4); break;     \
    case 5: CALL(5); break;     \
    default: return (int)hipErrorInvalidValue; \
  }

// a kernel over the launch's blocks of one kind, for one problem or a group
template <class KG, class KO, class... A>
int go(const QuadLaunch& L, const BlockMap* map, int grid, hipStream_t s, KG kg, KO ko, const QuadSys& S, A... a) {
  if (L.inst)
    kg<<<dim3(grid), dim3(kQuadThreads), 0, s>>>(S, SelGroup{L.inst, map}, a...);
  else
    ko<<<dim3(grid), dim3(kQuadThreads), 0, s>>>(S, SelOne{L.one}, a...);
  return (int)hipGetLastError();
}

}  // namespace

// R (rows a wavefront walks; a block's four wavefronts walk 4 R) is the
// smallest that lets every task run at once: blocks beyond what the chip
// holds would start when the others end, and the row below each block is
// read twice.
void quad_plan(int nx, int ny, int nt, QuadInst& I) {
  I.nx = nx;
  I.ny = ny;
  I.W = nx + 1;
  I.G = I.W * (ny + 1);
  I.ntiles = (I.G + 63) / 64;
  const int64_t slots = 256 * (nt == 2 ? 4 : (nt == 3 ? 3 : 2));
  for (I.R = 1;; ++I.R) {
    I.NG = (ny + kNW * I.R) / (kNW * I.R);  // ceil((ny + 1) / 4R)
    const int64_t t = ((int64_t)I.W * I.NG + kQuadOwn - 1) / kQuadOwn;
    I.tasks = (int)t;
    if (t <= slots || I.NG == 1) break;
  }
  I.nbM = (int)std::min<int64_t>(I.tasks, 2048);
  I.nbE = std::min((I.ntiles + kNW - 1) / kNW, 1024);
  I.nbQ = (int)(((int64_t)nx * ny + quads_per_block(nt) - 1) / quads_per_block(nt));
}

QuadLaunch quad_launch_one(const QuadInst& I, int nt) {
  QuadLaunch L;
  L.one = I;
  L.gM = I.nbM;
  L.gE = I.nbE;
  L.gQ = I.nbQ;
  return L;
}

double quad_omega_factor(int k) { return k % 2 ? 1.27 : 1.42; }

#define GO(KIND, K, ...) go(L, L.map##KIND, L.g##KIND, s, K<SelGroup>, K<SelOne>, S, ##__VA_ARGS__)
#define GO1(KIND, K, T1, ...) \
  go(L, L.map##KIND, L.g##KIND, s, K<T1, SelGroup>, K<T1, SelOne>, S, ##__VA_ARGS__)
#define GO2(KIND, K, T1, T2, ...) \
  go(L, L.map##KIND, L.g##KIND, s, K<T1, T2, SelGroup>, K<T1, T2, SelOne>, S, ##__VA_ARGS__)
#define QTRY(x)         \
  do {                  \
    const int e_ = (x); \
    if (e_) return e_;  \
  } while (0)

int launch_quad_clear(const QuadSys& S, const QuadLaunch& L, hipStream_t s) { return GO(E, q_clear_kernel); }

int launch_quad_build(const QuadSys& S, const QuadLaunch& L, hipStream_t s) {
  QTRY(GO(E, q_mask_kernel));
#define RUN(NT)                      \
  QTRY(GO1(Q, q_build_kernel, NT));  \
  QTRY(GO1(E, q_diag_kernel, NT));
  Q_NT(S.nt, RUN)
#undef RUN
  return 0;
}

int launch_quad_float(const QuadSys& S, hipStream_t s) {
  QTRY(launch_to_float(S.blk, S.fblk, S.tiles * 64 * quad_blk_vals(S.nt), s));
  QTRY(launch_to_float(S.Dinv, S.fDinv, S.tiles * 64 * quad_diag_vals(S.nt), s));
  return launch_to_float(S.tp, S.ftp, S.tiles * 64 * quad_tp_vals(S.nt), s);
}

int launch_quad_tp(const QuadSys& S, const QuadLaunch& L, hipStream_t s) {
#define RUN(NT) QTRY(GO1(E, q_tp_kernel, NT));
  Q_NT(S.nt, RUN)
#undef RUN
  return 0;
}

int launch_quad_l1(const QuadSys& S, const QuadLaunch& L, hipStream_t s) { return GO(E, q_l1_kernel); }

int launch_quad_omega(const QuadSys& S, const QuadLaunch& L, double factor, int steps, hipStream_t s) {
  steps = std::min(std::max(steps, 1), kLanczos);
#define INIT(NT) QTRY(GO2(E, q_init_kernel, NT, true));
#define PROD(NT) QTRY(GO2(M, q_product_kernel, NT, true, 0.0, steps, 0));
#define UPD(NT) QTRY(GO1(E, q_lupd_kernel, NT));
  Q_NT(S.nt, INIT)
  for (int i = 1; i <= steps; ++i) {
    Q_NT(S.nt, PROD)
    if (i < steps) Q_NT(S.nt, UPD)
  }
#undef INIT
#undef PROD
#undef UPD
  return go(L, nullptr, L.ninst, s, q_omega_kernel<SelGroup>, q_omega_kernel<SelOne>, S, steps, factor);
}

int launch_quad_init(const QuadSys& S, const QuadLaunch& L, hipStream_t s) {
#define INIT(NT) QTRY(GO2(E, q_init_kernel, NT, false));
  Q_NT(S.nt, INIT)
#undef INIT
  return 0;
}

namespace {
int product_t(const QuadSys& S, const QuadLaunch& L, double rtol2, int maxit, int force, hipStream_t s) {
#define PROD(NT) QTRY(GO2(M, q_product_kernel, NT, false, rtol2, maxit, force));
  Q_NT(S.nt, PROD)
#undef PROD
  return 0;
}
template <class W>
int residual_t(const QuadSys& S, const W* blk, const W* Dinv, const QuadLaunch& L, int force, hipStream_t s) {
#define RES(NT) QTRY(GO2(M, q_residual_kernel, NT, W, blk, Dinv, force));
  Q_NT(S.nt, RES)
#undef RES
  return 0;
}
template <class W>
int smooth_t(const QuadSys& S, const W* tp, const W* Dinv, const QuadLaunch& L, hipStream_t s) {
#define SMO(NT) QTRY(GO2(E, q_smooth_kernel, NT, W, tp, Dinv));
  Q_NT(S.nt, SMO)
#undef SMO
  return 0;
}
}  // namespace

int launch_quad_product(const QuadSys& S, const QuadLaunch& L, double rtol2, int maxit, hipStream_t s) {
  return product_t(S, L, rtol2, maxit, 0, s);
}
int launch_quad_residual(const QuadSys& S, const QuadLaunch& L, bool mixed, hipStream_t s) {
  return mixed ? residual_t<float>(S, S.fblk, S.fDinv, L, 0, s) : residual_t<double>(S, S.blk, S.Dinv, L, 0, s);
}
int launch_quad_smooth(const QuadSys& S, const QuadLaunch& L, bool mixed, hipStream_t s) {
  return mixed ? smooth_t<float>(S, S.ftp, S.fDinv, L, s) : smooth_t<double>(S, S.tp, S.Dinv, L, s);
}
int launch_quad_finish(const QuadSys& S, const QuadLaunch& L, double* uhat, double* out, hipStream_t s) {
  const int resid = out && !S.from_k ? 1 : 0;
#define FIN(NT) QTRY(GO1(Q, q_finish_kernel, NT, uhat, resid));
  Q_NT(S.nt, FIN)
#undef FIN
  if (!resid) return 0;
#define NRM(NT) QTRY(GO1(E, q_resnorm_kernel, NT));
  Q_NT(S.nt, NRM)
#undef NRM
  return go(L, nullptr, L.ninst, s, q_sum_kernel<SelGroup>, q_sum_kernel<SelOne>, S, out);
}

int launch_quad_time(const QuadSys& S, const QuadLaunch& L, int which, hipStream_t s) {
  return which == 1 ? residual_t<double>(S, S.blk, S.Dinv, L, 1, s) : product_t(S, L, 0.0, 0, 1, s);
}

}  // namespace hdg
