// Static condensation (examples/poisson2D_HDG.jl:155-174) through the Schur
// complement on the u block, for kappa = 1 and a reference mass that the
// quadrature leaves SPD (k = 1 at degree 2, k = 3 at degree 6, k <= 2 at
// degree 4).
//
// With Me = [A -B; B' C], EFe = [-E; F], Bte = [0; be] and A = detJ
// diag(Mref, Mref) on an affine cell:
//   S   = C + B' A^-1 B                      (nu x nu, SPD)
//   R   = F + B' A^-1 E,  U = S^-1 R,  Q = A^-1 (B U - E)     K_e = [Q; U]
//   Ub  = S^-1 be,  Qb = A^-1 B Ub                            b_e = [Qb; Ub]
//   Ate = E'Q + F'U - H = R' S^-1 R - E' A^-1 E - H
//   bte = -(E'Qb + F'Ub) = -R' S^-1 be
// Every product through A^-1 is a combination of constant reference
// matrices (SpdLayout, hdg_tables.h) with the metric detJ J^-1 J^-T, the
// scaled normals J^-1 n |e| and the edge lengths, so a cell costs a 10 x 10
// Cholesky factorisation (k = 3) and small matrix-vector products instead of
// the elimination of its 30 x 30 local matrix.
//
// Mapping: four lanes per element (16 per wavefront), a DPP quad.  Every lane
// forms S and factors it in registers; lanes 0..2 carry the nt trace columns
// of their face, one after another, lane 3 the rhs column.  The columns
// Y = L^-1 R meet in LDS for the products of Ate.
#include <hip/hip_runtime.h>

#include "hdg_device.h"
#include "hdg_internal.h"

namespace hdg {

namespace {

template <int K>
struct SpdDims {
  static constexpr int NU = (K + 1) * (K + 2) / 2, NQ = 2 * NU, M = 3 * NU, NT = K + 1, NTR = 3 * NT;
  static constexpr int NL = NU * (NU + 1) / 2;  // packed lower triangle
  static constexpr int YS = NU * (NTR + 1) + NTR;  // LDS of one element: L^-1 [R be], Ate c
  // tables staged in LDS: Gam, Z, then Om to the end
  static constexpr int T1 = 18 * NU * NT;
  // table offsets (SpdLayout; the quadrature tables Nw, Mg follow at Nw)
  static constexpr int R = 0, C = 3 * NU * NU, Gam = 6 * NU * NU, Z = Gam + 6 * NU * NT, V = Z + 12 * NU * NT,
                       P = V + 6 * NU * NT, Om = P + 2 * NU * NU, H = Om + 36 * NT * NT, Nw = H + NT * NT;
};

constexpr int kSeg = 16;  // lanes per element of the recovery
constexpr int kCells = 64;  // elements per block of the condensation

__host__ __device__ constexpr int tri(int i, int j) { return i * (i + 1) / 2 + j; }  // i >= j

// Tables read at compile-time offsets by every lane alike: through the scalar
// cache, as operands that cost no vector register and no LDS.
typedef const double __attribute__((address_space(4))) * ScalarTab;

// WPE: waves per SIMD the register budget is cut for (2: none spilled at k <=
// 2, 80 B per lane at k = 3; 3: 440 B at k = 3, 5.5 ms at 1024^2); 2 by
// default, or the autotuner's choice.  The LDS of a block (spd_lds) decides how
// many waves there are: 84,448 B at k = 3 and degree 6, one block of the CU's
// 163,840 B and one wave per SIMD.
// GROUPED: several instances packed into one mesh, the source of cell c is
// srcs[cell_inst[c]].
//
// Bound by its stores (Ate, the u rows, 2.3 KB per cell at k = 3: 0.95 ms for
// 1024^2 grid cells at the rate of a copy) and the issue of the products
// beside them, at k = 3 from one wave per SIMD: 2.9 ms there, 0.29 at 768^2,
// k = 1.
// With 16 lanes per element, one column each, the factor in LDS and every
// table read from LDS by every element: 5.9 and 0.58 ms.
template <int K, int WPE, bool GROUPED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE)))
void condense_spd_kernel(CondenseArgs a) {
  using D = SpdDims<K>;
  constexpr int NU = D::NU, M = D::M, NT = D::NT, NTR = D::NTR, NL = D::NL;
  extern __shared__ __align__(16) double sh[];
  const SpdLayoutDev L = a.spd;
  const int tail = L.total - D::Om;
  for (int i = threadIdx.x; i < D::T1; i += 256) sh[i] = a.spd_tables[D::Gam + i];
  for (int i = threadIdx.x; i < tail; i += 256) sh[D::T1 + i] = a.spd_tables[D::Om + i];
  __syncthreads();
  const double* const TG = sh;                       // Gam
  const double* const TZ = sh + 6 * NU * NT;         // Z
  const double* const TO = sh + D::T1;               // Om
  const double* const TH = TO + 36 * NT * NT;        // H
  const double* const TN = TO + (D::Nw - D::Om);     // Nw, Mg

  const int l = threadIdx.x & 3, slot = threadIdx.x >> 2;
  double* const Y = sh + ((D::T1 + tail + 1) & ~1) + slot * D::YS;
  double* const Rv = Y + NU * (NTR + 1);
  const int64_t count = a.mesh.nc;
  const int nqp = L.nqp;
  const double tau = a.tau;
  const int fl = l < 3 ? l : 0;

  for (int64_t base = (int64_t)blockIdx.x * kCells; base < count; base += (int64_t)gridDim.x * kCells) {
    const bool valid = base + slot < count;
    const int64_t cell = valid ? base + slot : count - 1;
    Geo g;
    cell_geometry(a.mesh, cell, g);
    const SrcParams& S = GROUPED ? a.srcs[a.cell_inst[cell]] : a.src;

    // be_i = sum_q w_q N_i(q) detJ f(x_q): the lanes share the points
    double rb[NU];
#pragma unroll
    for (int i = 0; i < NU; ++i) rb[i] = 0.0;
    for (int q = l; q < nqp; q += 4) {
      double xq = 0.0, yq = 0.0;
#pragma unroll
      for (int v = 0; v < 3; ++v) {
        xq += TN[NU * nqp + v * nqp + q] * g.x[2 * v];
        yq += TN[NU * nqp + v * nqp + q] * g.x[2 * v + 1];
      }
      const double fv = g.detJ * (S.kind == 3 ? __ldg(S.f_qp + cell + a.mesh.nc * (int64_t)q) : Src::f(S, xq, yq));
#pragma unroll
      for (int i = 0; i < NU; ++i) rb[i] = fma(TN[i * nqp + q], fv, rb[i]);
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      rb[i] += dpp_quad<0xB1>(rb[i]);
      rb[i] += dpp_quad<0x4E>(rb[i]);
    }
    __builtin_amdgcn_sched_barrier(0);

    // the lane's face: length, unit normal, orientation (blended, so that
    // the lane-dependent choice does not index the geometry)
    const double w0 = (double)(fl == 0), w1 = (double)(fl == 1), w2 = (double)(fl == 2);
    const double el = w0 * g.len[0] + w1 * g.len[1] + w2 * g.len[2];
    const double nx = w0 * g.nrm[0] + w1 * g.nrm[2] + w2 * g.nrm[4];
    const double ny = w0 * g.nrm[1] + w1 * g.nrm[3] + w2 * g.nrm[5];
    const int of = (fl == 0) * g.ori[0] + (fl == 1) * g.ori[1] + (fl == 2) * g.ori[2];
    const int fo = fl * 2 + of;

    // S = tau sum_f |e_f| Cref_f + detJ (G00 R00 + G01 R01 + G11 R11),
    // G = J^-1 J^-T, and S = L L' in place (1 / L_ii on the diagonal)
    double Lr[NL];
    bool bad = !(g.detJ > 0.0);
    {
      const double c0 = tau * g.len[0], c1 = tau * g.len[1], c2 = tau * g.len[2];
      const double r0 = g.detJ * (g.Ji[0] * g.Ji[0] + g.Ji[2] * g.Ji[2]);
      const double r1 = g.detJ * (g.Ji[0] * g.Ji[1] + g.Ji[2] * g.Ji[3]);
      const double r2 = g.detJ * (g.Ji[1] * g.Ji[1] + g.Ji[3] * g.Ji[3]);
      double dmax = 0.0;
      // the tables' address is renewed row by row: loop-invariant to the
      // compiler, all of their values would be kept (in spilled registers)
      uintptr_t tab = (uintptr_t)a.spd_tables;
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        asm volatile("" : "+s"(tab));
        const ScalarTab TS = (ScalarTab)tab;
#pragma unroll
        for (int j = 0; j <= i; ++j) {
          const int x = i * NU + j;
          Lr[tri(i, j)] = c0 * TS[D::C + x] + c1 * TS[D::C + NU * NU + x] + c2 * TS[D::C + 2 * NU * NU + x] +
                          r0 * TS[D::R + x] + r1 * TS[D::R + NU * NU + x] + r2 * TS[D::R + 2 * NU * NU + x];
          if (j % 2) __builtin_amdgcn_sched_barrier(0);
        }
        dmax = fmax(dmax, Lr[tri(i, i)]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < NU; ++i) {
        double d = Lr[tri(i, i)];
#pragma unroll
        for (int j = 0; j < i; ++j) {
          double v = Lr[tri(i, j)];
#pragma unroll
          for (int t = 0; t < j; ++t) v -= Lr[tri(i, t)] * Lr[tri(j, t)];
          v *= Lr[tri(j, j)];
          Lr[tri(i, j)] = v;
          d -= v * v;
          __builtin_amdgcn_sched_barrier(0);
        }
        bad |= !(d > 1e-10 * dmax);
        Lr[tri(i, i)] = 1.0 / (d > 0.0 ? sqrt(d) : 1.0);
      }
    }

    // the columns Y = L^-1 R into LDS; trace column: R = tau |e_f| Gam_fo +
    // s0 Z_0fo + s1 Z_1fo with s_d = |e_f| (J^-1 n_f)_d
    {
      const double s0 = el * (g.Ji[0] * nx + g.Ji[2] * ny), s1 = el * (g.Ji[1] * nx + g.Ji[3] * ny);
      const double tf = tau * el;
#pragma unroll 1
      for (int t = 0; t < NT; ++t) {
        double rc[NU];
#pragma unroll
        for (int i = 0; i < NU; ++i) {
          const double v = tf * TG[(fo * NU + i) * NT + t] + s0 * TZ[(fo * NU + i) * NT + t] +
                           s1 * TZ[((6 + fo) * NU + i) * NT + t];
          rc[i] = l < 3 ? v : rb[i];
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < NU; ++i) {
          double v = rc[i];
#pragma unroll
          for (int u = 0; u < i; ++u) v -= Lr[tri(i, u)] * rc[u];
          rc[i] = v * Lr[tri(i, i)];
        }
        double* const y = Y + (l < 3 ? l * NT + t : NTR) * NU;
#pragma unroll
        for (int i = 0; i < NU; ++i) y[i] = rc[i];
        // U = L^-T Y: the u rows of K_e (trace columns) and of b_e (rhs
        // column), compact at the start of the cell's K_e and b_e blocks (U
        // column-major nu x ntr); the q rows Q = A^-1 (B U - E) follow from
        // them and the cell's geometry, and are formed where they are needed
        // (recover_spd_kernel for the recovered q, expand_ke_spd_kernel for
        // hdg_get_local_ops, which also restores the layout of K_e)
#pragma unroll
        for (int i = NU - 1; i >= 0; --i) {
          double v = rc[i];
#pragma unroll
          for (int u = i + 1; u < NU; ++u) v -= Lr[tri(u, i)] * rc[u];
          rc[i] = v * Lr[tri(i, i)];
        }
        if (valid && (l < 3 || t == 0)) {
          double* out = l < 3 ? a.Ke + cell * (int64_t)(M * NTR) + (l * NT + t) * NU : a.be + cell * (int64_t)M;
          if constexpr (NU % 2 == 0) {
#pragma unroll
            for (int i = 0; i < NU; i += 2) *reinterpret_cast<double2*>(out + i) = make_double2(rc[i], rc[i + 1]);
          } else {
#pragma unroll
            for (int i = 0; i < NU; ++i) out[i] = rc[i];
          }
        }
      }
    }
    // an element's lanes are of one wavefront, whose LDS instructions run in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // Ate = Y'Y - E'A^-1 E - H and bte = -Y' y_b, column by column (Ate is
    // symmetric: column s is stored as row s).  E'A^-1 E entry ((f,t),(g,s)) =
    // |e_f| |e_g| (n_f . n_g) / detJ Om_fo,gp(t,s).
    //
    // Constant traces: for c = 1 on mode 0 of every face the local problem is
    // solved by u = const, q = 0, so in exact arithmetic Ate c = F'u - H c =
    // (tau - 1) H c (H carries no tau, poisson2D_HDG.jl:149).  The rounding of
    // the shared tables breaks this the same way in every cell, an error the
    // trace solve amplifies by cond(K) ~ h^-2 (1024^2 cells, P3: an L2 error
    // of 6e-10 instead of 5e-13).  Ate is projected onto it, with d = Ate c -
    // (tau - 1) H c:
    //   Ate - (d c' + c d') / 3 + (c'd) c c' / 9,
    // a symmetric change of the order of the rounding (~1e-15 relative).  The
    // columns of modes t > 0 need their own d only, those of mode 0 all of it:
    // t runs down, d through LDS.
    const double sc = el / g.detJ;
    const double cg[3] = {sc * g.len[0] * (nx * g.nrm[0] + ny * g.nrm[1]),
                          sc * g.len[1] * (nx * g.nrm[2] + ny * g.nrm[3]),
                          sc * g.len[2] * (nx * g.nrm[4] + ny * g.nrm[5])};
#pragma unroll 1
    for (int t = NT - 1; t >= 0; --t) {
      double y[NU], row[NTR];
      // an offset the compiler takes as new from column to column: it would
      // load all columns ahead, and hold them across the loop, otherwise
      int o = 0;
      asm volatile("" : "+v"(o));
      const double* yo = Y + o + (l < 3 ? l * NT + t : NTR) * NU;
#pragma unroll
      for (int i = 0; i < NU; ++i) y[i] = yo[i];
#pragma unroll
      for (int gs = 0; gs < 3; ++gs) {
        const double* om = TO + ((fo * 6 + gs * 2 + g.ori[gs]) * NT + t) * NT;
        const double hl = gs == fl ? el : 0.0;
#pragma unroll
        for (int us = 0; us < NT; ++us) {
          const double* ys = Y + o + (gs * NT + us) * NU;
          double dot = 0.0;
#pragma unroll
          for (int i = 0; i < NU; ++i) dot = fma(ys[i], y[i], dot);
          if ((gs * NT + us) % 2) asm volatile("" : "+v"(o), "+v"(dot));
          row[gs * NT + us] = dot - cg[gs] * om[us] - hl * TH[t * NT + us];
        }
      }
      double bt = 0.0;
#pragma unroll
      for (int i = 0; i < NU; ++i) bt = fma(Y[o + NTR * NU + i], y[i], bt);
      const double d = ((row[0] + row[NT]) + row[2 * NT]) - (tau - 1.0) * el * TH[t * NT];
      if (t > 0) {
        if (l < 3) Rv[l * NT + t] = d;
#pragma unroll
        for (int gs = 0; gs < 3; ++gs) row[gs * NT] -= d * (1.0 / 3.0);
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const double d0[3] = {dpp_quad<0x00>(d), dpp_quad<0x55>(d), dpp_quad<0xAA>(d)};
        const double ds = (d0[0] + d0[1] + d0[2]) * (1.0 / 9.0);
#pragma unroll
        for (int gs = 0; gs < 3; ++gs) {
          row[gs * NT] += ds - (d + d0[gs]) * (1.0 / 3.0);
#pragma unroll
          for (int us = 1; us < NT; ++us) row[gs * NT + us] -= Rv[gs * NT + us] * (1.0 / 3.0);
        }
      }
      if (valid && l < 3) {
        double* at = a.Ate + cell * (int64_t)(NTR * NTR) + (l * NT + t) * NTR;
        if constexpr (NTR % 2 == 0) {
#pragma unroll
          for (int s = 0; s < NTR; s += 2) *reinterpret_cast<double2*>(at + s) = make_double2(row[s], row[s + 1]);
        } else {
#pragma unroll
          for (int s = 0; s < NTR; ++s) at[s] = row[s];
        }
        a.bte[cell * NTR + l * NT + t] = -bt;
      }
    }
    if (valid && bad && l == 0) atomicOr(a.err + (GROUPED ? a.cell_inst[cell] : 0), g.detJ > 0.0 ? 2 : 1);
    __builtin_amdgcn_wave_barrier();
  }
}

// K_e and b_e in their exported layout (column t of K_e: q rows then u rows)
// from the compact u rows the Schur kernel stores (U column-major at the
// start of the cell's block, Ub at the start of b_e's), with the q rows
//   Q_t = A^-1 (B U_t - E_t) = sum_d (J^-1)_dc P_d U_t - |e_f| n_fc / detJ V_fo(:, s)
// for trace column t = (face f, mode s), without the E term for the rhs.
// One thread per cell, in place: column t (written at t m) reads compact
// column t (at t nu) before writing, and the columns run from the last, so
// every compact column a write covers has been read already.  Tables
// staged in LDS.
template <int K>
__global__ __launch_bounds__(256) void expand_ke_spd_kernel(DevMesh m, const double* __restrict__ tab,
                                                            double* __restrict__ Ke, double* __restrict__ be) {
  using D = SpdDims<K>;
  constexpr int NU = D::NU, NQ = D::NQ, M = D::M, NT = D::NT, NTR = D::NTR;
  __shared__ double T[D::Om - D::V];  // V then P
  for (int i = threadIdx.x; i < D::Om - D::V; i += blockDim.x) T[i] = __ldg(tab + D::V + i);
  __syncthreads();
  const double* V = T;
  const double* Pm = T + (D::P - D::V);
  const int64_t cell = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= m.nc) return;
  Geo g;
  cell_geometry(m, cell, g);
  double* ke = Ke + cell * (int64_t)(M * NTR);
#pragma unroll 1
  for (int col = NTR; col >= 0; --col) {
    // col == NTR: the rhs column (b_e)
    const double* in = col < NTR ? ke + col * NU : be + cell * (int64_t)M;
    double* out = col < NTR ? ke + col * M : be + cell * (int64_t)M;
    double u[NU];
#pragma unroll
    for (int i = 0; i < NU; ++i) u[i] = in[i];
    const int fl = col < NTR ? col / NT : 0, tl = col < NTR ? col - fl * NT : 0;
    const double el = g.len[fl];
    const double nx = g.nrm[2 * fl], ny = g.nrm[2 * fl + 1];
    const int fo = fl * 2 + g.ori[fl];
    const double vs = col < NTR ? el / g.detJ : 0.0;
#pragma unroll 1
    for (int i = 0; i < NU; ++i) {
      double t0 = 0.0, t1 = 0.0;
#pragma unroll
      for (int j = 0; j < NU; ++j) {
        t0 += Pm[i * NU + j] * u[j];
        t1 += Pm[(NU + i) * NU + j] * u[j];
      }
      const double v = vs * V[(fo * NU + i) * NT + tl];
      out[i] = g.Ji[0] * t0 + g.Ji[1] * t1 - nx * v;
      out[NU + i] = g.Ji[2] * t0 + g.Ji[3] * t1 - ny * v;
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) out[NQ + i] = u[i];
  }
}

// Recovery (examples/poisson2D_HDG.jl:197-212) from the u rows of K_e:
// u = U uhat_c + Ub, q = sum_d (J^-1)_dc P_d u - sum_f |e_f| n_fc / detJ
// V_fo uhat_f, i.e. K_e uhat_c + b_e with the q rows applied to the one
// trace vector.  16 lanes per cell (4 per wavefront): lane i < nu forms
// u_i (reading row i of U: the lanes of a cell read runs of nu doubles),
// then q_i from u, which the lanes of the cell exchange by shuffles.
// Tables staged in LDS.
template <int K>
__global__ __launch_bounds__(256) void recover_spd_kernel(DevMesh m, const double* __restrict__ tab,
                                                          const double* __restrict__ Ke,
                                                          const double* __restrict__ be,
                                                          const double* __restrict__ uhat, double* __restrict__ qu) {
  using D = SpdDims<K>;
  constexpr int NU = D::NU, NQ = D::NQ, M = D::M, NT = D::NT, NTR = D::NTR;
  static_assert(NU <= kSeg, "segment too small");
  __shared__ double T[D::Om - D::V];  // V then P
  for (int i = threadIdx.x; i < D::Om - D::V; i += blockDim.x) T[i] = __ldg(tab + D::V + i);
  __syncthreads();
  const double* V = T;
  const double* Pm = T + (D::P - D::V);
  const int lane = threadIdx.x & 63;
  const int sbase = (lane / kSeg) * kSeg, ls = lane - sbase;
  // every lane of a segment has the same cell: segments leave together
  const int64_t cell = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kSeg;
  if (cell >= m.nc) return;
  Geo g;
  cell_geometry(m, cell, g);
  double uh[NTR];
#pragma unroll
  for (int lf = 0; lf < 3; ++lf) {
    const int64_t f = m.cf[3 * cell + lf];
#pragma unroll
    for (int b = 0; b < NT; ++b) uh[lf * NT + b] = uhat[f * NT + b];
  }
  const int i = ls < NU ? ls : NU - 1;  // lanes past nu repeat the last row and store nothing
  // the compact u rows: U column-major (nu x ntr) at the start of the cell's
  // K_e block, Ub at the start of its b_e block
  const double* ke = Ke + cell * (int64_t)(M * NTR) + i;
  double u = be[cell * M + i];
#pragma unroll
  for (int t = 0; t < NTR; ++t) u = fma(ke[t * NU], uh[t], u);
  double wx = 0.0, wy = 0.0;
#pragma unroll
  for (int lf = 0; lf < 3; ++lf) {
    const double sc = g.len[lf] / g.detJ;
    const double sx = sc * g.nrm[2 * lf], sy = sc * g.nrm[2 * lf + 1];
    const int fo = lf * 2 + g.ori[lf];
    double v = 0.0;
#pragma unroll
    for (int b = 0; b < NT; ++b) v = fma(V[(fo * NU + i) * NT + b], uh[lf * NT + b], v);
    wx = fma(sx, v, wx);
    wy = fma(sy, v, wy);
  }
  double t0 = 0.0, t1 = 0.0;
#pragma unroll
  for (int j = 0; j < NU; ++j) {
    const double uj = __shfl(u, sbase + j, 64);
    t0 = fma(Pm[i * NU + j], uj, t0);
    t1 = fma(Pm[(NU + i) * NU + j], uj, t1);
  }
  if (ls < NU) {
    double* o = qu + cell * (int64_t)M;
    o[i] = g.Ji[0] * t0 + g.Ji[1] * t1 - wx;
    o[NU + i] = g.Ji[2] * t0 + g.Ji[3] * t1 - wy;
    o[NQ + i] = u;
  }
}

// LDS bytes of a block of the condensation
template <int K>
size_t spd_lds(const SpdLayoutDev& L) {
  using D = SpdDims<K>;
  return sizeof(double) * (((D::T1 + L.total - D::Om + 1) & ~1) + kCells * D::YS);
}
// blocks on a CU by their LDS, a wave per SIMD each
constexpr size_t kLdsPerCu = 160u << 10;
int spd_waves(int k, const SpdLayoutDev& L) {
  return (int)(kLdsPerCu / (k == 1 ? spd_lds<1>(L) : (k == 2 ? spd_lds<2>(L) : spd_lds<3>(L))));
}

template <int K>
int spd_launch(const CondenseArgs& a, int wpe, int grid_cap, hipStream_t s) {
  using D = SpdDims<K>;
  // the kernel addresses the constant tables at compile-time offsets
  const SpdLayoutDev& L = a.spd;
  if (L.nu != D::NU || L.nt != D::NT || L.R != D::R || L.C != D::C || L.Gam != D::Gam || L.Z != D::Z ||
      L.V != D::V || L.P != D::P || L.Om != D::Om || L.H != D::H || L.Nw != D::Nw ||
      L.Mg != D::Nw + D::NU * L.nqp || L.total != L.Mg + 3 * L.nqp)
    return (int)hipErrorInvalidValue;
  const int64_t n = a.mesh.nc;
  int64_t grid = (n + kCells - 1) / kCells;
  const int64_t cap = grid_cap > 0 ? grid_cap : 16384;
  if (grid < 1) grid = 1;
  if (grid > cap) grid = cap;
  const size_t lds = spd_lds<K>(L);
  if (wpe != 3) wpe = 2;
  if (a.srcs) {
    if (wpe == 2)
      hipLaunchKernelGGL((condense_spd_kernel<K, 2, true>), dim3((int)grid), dim3(256), lds, s, a);
    else
      hipLaunchKernelGGL((condense_spd_kernel<K, 3, true>), dim3((int)grid), dim3(256), lds, s, a);
  } else {
    if (wpe == 2)
      hipLaunchKernelGGL((condense_spd_kernel<K, 2, false>), dim3((int)grid), dim3(256), lds, s, a);
    else
      hipLaunchKernelGGL((condense_spd_kernel<K, 3, false>), dim3((int)grid), dim3(256), lds, s, a);
  }
  return (int)hipGetLastError();
}

}  // namespace

int launch_condense_spd(int k, const CondenseArgs& a, const CondenseSched& sc, hipStream_t s) {
  if (!a.spd_tables) return (int)hipErrorInvalidValue;
  switch (k) {
    case 1: return spd_launch<1>(a, sc.spd_wpe, sc.spd_grid, s);
    case 2: return spd_launch<2>(a, sc.spd_wpe, sc.spd_grid, s);
    case 3: return spd_launch<3>(a, sc.spd_wpe, sc.spd_grid, s);
    default: return (int)hipErrorInvalidValue;
  }
}

int launch_recover_spd(int k, const DevMesh& m, const double* tab, const double* Ke, const double* be,
                       const double* uhat, double* qu, hipStream_t s) {
  const int64_t g = (m.nc * kSeg + 255) / 256;
  const dim3 grid((unsigned)(g > 0 ? g : 1));
  switch (k) {
    case 1: hipLaunchKernelGGL(recover_spd_kernel<1>, grid, dim3(256), 0, s, m, tab, Ke, be, uhat, qu); break;
    case 2: hipLaunchKernelGGL(recover_spd_kernel<2>, grid, dim3(256), 0, s, m, tab, Ke, be, uhat, qu); break;
    case 3: hipLaunchKernelGGL(recover_spd_kernel<3>, grid, dim3(256), 0, s, m, tab, Ke, be, uhat, qu); break;
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}

int launch_expand_ke_spd(int k, const DevMesh& m, const double* tab, double* Ke, double* be, hipStream_t s) {
  const int64_t g = (m.nc + 255) / 256;
  const dim3 grid((unsigned)(g > 0 ? g : 1));
  switch (k) {
    case 1: hipLaunchKernelGGL(expand_ke_spd_kernel<1>, grid, dim3(256), 0, s, m, tab, Ke, be); break;
    case 2: hipLaunchKernelGGL(expand_ke_spd_kernel<2>, grid, dim3(256), 0, s, m, tab, Ke, be); break;
    case 3: hipLaunchKernelGGL(expand_ke_spd_kernel<3>, grid, dim3(256), 0, s, m, tab, Ke, be); break;
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}

int tune_condense_spd(int k, const CondenseArgs& a, hipStream_t s, CondenseSched* best, double* best_us,
                      double* default_us) {
  hipEvent_t e0, e1;
  hipError_t e = hipEventCreate(&e0);
  if (e != hipSuccess) return (int)e;
  e = hipEventCreate(&e1);
  if (e != hipSuccess) {
    (void)hipEventDestroy(e0);
    return (int)e;
  }
  const int grids[] = {2048, 4096, 8192, 16384};
  constexpr int kReps = 3;
  double bt = 1e300, dt = 0.0;
  CondenseSched bs = *best;
  int rc = 0;
  // the narrow register budget only where three blocks fit on a CU
  for (int wpe = spd_waves(k, a.spd) >= 3 ? 3 : 2; wpe >= 2 && rc == 0; --wpe)
    for (int g : grids) {
      CondenseSched sc = *best;
      sc.spd_wpe = wpe;
      sc.spd_grid = g;
      rc = launch_condense_spd(k, a, sc, s);  // warm-up
      if (rc) break;
      (void)hipEventRecord(e0, s);
      for (int r = 0; r < kReps && rc == 0; ++r) rc = launch_condense_spd(k, a, sc, s);
      (void)hipEventRecord(e1, s);
      if (rc || (rc = (int)hipEventSynchronize(e1))) break;
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, e0, e1);
      const double us = 1e3 * ms / kReps;
      if (us < bt) {
        bt = us;
        bs = sc;
      }
      if (wpe == 2 && g == 16384) dt = us;
    }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  *best = bs;
  if (best_us) *best_us = bt;
  if (default_us) *default_us = dt;
  return 0;
}

}  // namespace hdg
