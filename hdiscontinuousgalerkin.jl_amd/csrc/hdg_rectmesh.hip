// rectangle_mesh(TriangleCell, (nx, ny), LL, UR) generated on the device
// (src/generate_mesh.jl:1-18,110-143): the same node coordinates,
// cells, face numbering and boundary classification as the host generator
// (hdg_mesh.cpp), bit for bit, plus the structures the solver derives from
// them (face end points, vertex -> face lists, the four vertices around each
// face) in closed form.  Coordinates are rounded operation by operation,
// as the host file is compiled without FMA contraction: contraction is off
// for this file (device code otherwise contracts a * b + c into one fma).
#include <hip/hip_runtime.h>

#include "hdg_internal.h"

#pragma clang fp contract(off)

namespace hdg {

namespace {

__device__ inline uint64_t splitmix64_d(uint64_t z) {
  z += 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}

// 1-based ids of the faces first created by grid cell (i, j), in the order
// rectangle_mesh meets them: diagonal, left, bottom of the lower triangle;
// top, right of the upper one (the closed form of hdg_mesh.cpp's sweep).
struct SweepD {
  int64_t nx, ny;
  __device__ int64_t base(int64_t j) const { return j == 1 ? 0 : (4 * nx + 1) + (j - 2) * (3 * nx + 1); }
  __device__ int64_t D(int64_t i, int64_t j) const {
    if (i == 1) return base(j) + 1;
    return base(j) + (j == 1 ? 5 + 4 * (i - 2) : 4 + 3 * (i - 2)) + 1;
  }
  __device__ int64_t T(int64_t i, int64_t j) const {
    if (j == 1) return i == 1 ? base(j) + 4 : base(j) + 5 + 4 * (i - 2) + 3;
    return i == 1 ? base(j) + 3 : base(j) + 4 + 3 * (i - 2) + 2;
  }
  __device__ int64_t R(int64_t i, int64_t j) const {
    if (j == 1) return i == 1 ? base(j) + 5 : base(j) + 5 + 4 * (i - 2) + 4;
    return i == 1 ? base(j) + 4 : base(j) + 4 + 3 * (i - 2) + 3;
  }
  __device__ int64_t L(int64_t i, int64_t j) const { return i == 1 ? base(j) + 2 : R(i - 1, j); }
  __device__ int64_t B(int64_t i, int64_t j) const {
    if (j > 1) return T(i, j - 1);
    return i == 1 ? base(j) + 3 : base(j) + 5 + 4 * (i - 2) + 2;
  }
};

// a (1 - r) + r b, rounded as the host evaluates it (no contraction here)
__device__ inline double lerp_rn(double a, double b, double r) { return a * (1.0 - r) + r * b; }

// node coordinates, then the jitter of interior nodes
__global__ void rm_nodes_kernel(RectMeshArgs a) {
  const int64_t nnx = a.nx + 1, nny = a.ny + 1;
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nnx * nny) return;
  const int64_t i = v / nnx, j = v % nnx;  // row, column (0-based), as the host loops
  const double rb = (double)i / (double)(nny - 1);
  const double xa = lerp_rn(a.x0, a.x0, rb), xb = lerp_rn(a.x1, a.x1, rb);
  const double ya = lerp_rn(a.y0, a.y1, rb), yb = lerp_rn(a.y0, a.y1, rb);
  const double ratio = (double)j / (double)(nnx - 1);
  double x = lerp_rn(xa, xb, ratio), y = lerp_rn(ya, yb, ratio);
  if (a.jitter > 0.0 && i >= 1 && i < a.ny && j >= 1 && j < a.nx) {
    const double hx = (a.x1 - a.x0) / (double)a.nx, hy = (a.y1 - a.y0) / (double)a.ny;
    const uint64_t n = (uint64_t)v;
    const double ux = (double)(splitmix64_d(a.seed + 2 * n) >> 11) * (1.0 / 9007199254740992.0);
    const double uy = (double)(splitmix64_d(a.seed + 2 * n + 1) >> 11) * (1.0 / 9007199254740992.0);
    x = x + a.jitter * hx * (2.0 * ux - 1.0);
    y = y + a.jitter * hy * (2.0 * uy - 1.0);
  }
  a.xy[2 * (a.node0 + v)] = x;
  a.xy[2 * (a.node0 + v) + 1] = y;
}

// cells (nodes, faces) of grid cell (i, j) and the faces it creates
__global__ void rm_cells_kernel(RectMeshArgs a) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= a.nx * a.ny) return;
  const int64_t i = g % a.nx + 1, j = g / a.nx + 1;
  const int64_t nnx = a.nx + 1;
  const SweepD S{a.nx, a.ny};
  auto node = [&](int64_t ii, int64_t jj) { return a.node0 + ii + (jj - 1) * nnx - 1; };  // 0-based, shifted
  const int64_t lo = 2 * ((j - 1) * a.nx + (i - 1)), up = lo + 1;  // 0-based, local
  const int64_t cl = a.cell0 + lo, cu = a.cell0 + up;
  const int64_t fD = S.D(i, j), fT = S.T(i, j), fR = S.R(i, j), fL = S.L(i, j), fB = S.B(i, j);
  int* cn = a.cn;
  int* cf = a.cf;
  cn[3 * cl] = (int)node(i, j);
  cn[3 * cl + 1] = (int)node(i + 1, j);
  cn[3 * cl + 2] = (int)node(i, j + 1);
  cf[3 * cl] = (int)(a.face0 + fD - 1);
  cf[3 * cl + 1] = (int)(a.face0 + fL - 1);
  cf[3 * cl + 2] = (int)(a.face0 + fB - 1);
  cn[3 * cu] = (int)node(i + 1, j);
  cn[3 * cu + 1] = (int)node(i + 1, j + 1);
  cn[3 * cu + 2] = (int)node(i, j + 1);
  cf[3 * cu] = (int)(a.face0 + fT - 1);
  cf[3 * cu + 1] = (int)(a.face0 + fD - 1);
  cf[3 * cu + 2] = (int)(a.face0 + fR - 1);
  if (a.cell_inst) {
    a.cell_inst[cl] = a.inst;
    a.cell_inst[cu] = a.inst;
  }
  // cells c1, c2 (0-based, global; -1 none) of face f (1-based, local)
  auto setf = [&](int64_t f, int64_t c1, int64_t c2) {
    const int64_t F = a.face0 + f - 1;
    a.fcell[2 * F] = (int)c1;
    a.fcell[2 * F + 1] = (int)c2;
  };
  setf(fD, cl, cu);
  if (i == 1) setf(fL, cl, -1);
  if (j == 1) setf(fB, cl, -1);
  setf(fT, cu, j < a.ny ? a.cell0 + 2 * (j * a.nx + (i - 1)) : -1);
  setf(fR, cu, i < a.nx ? a.cell0 + 2 * ((j - 1) * a.nx + i) : -1);
}

// A face with one cell must lie on a side of the box: both end points on
// the bottom, right, top or left side, by exact coordinate equality
// (_get_rectangular_boundary_sets, generate_mesh.jl:60-89); else bit 4 of
// the error flag (HDG_ERR_BOUNDARY on the host).
__global__ void rm_faces_kernel(RectMeshArgs a) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= a.nf) return;
  const int64_t F = a.face0 + f;
  if (a.fcell[2 * F + 1] >= 0) return;
  const int64_t c = a.fcell[2 * F];
  const int l = a.cf[3 * c] == F ? 0 : (a.cf[3 * c + 1] == F ? 1 : 2);
  const double *p = a.xy + 2 * (int64_t)a.cn[3 * c + (l + 1) % 3], *q = a.xy + 2 * (int64_t)a.cn[3 * c + (l + 2) % 3];
  const bool ok = (p[1] == a.y0 && q[1] == a.y0) || (p[0] == a.x1 && q[0] == a.x1) ||
                  (p[1] == a.y1 && q[1] == a.y1) || (p[0] == a.x0 && q[0] == a.x0);
  if (!ok) atomicOr(a.err, 4);
}

// Every dof of every face with one cell is prescribed, the others are free.
// u = value on the boundary: the trace basis is the orthonormal Legendre
// basis on [0, 1] with P0 = 1, so the projection of a constant is `value`
// on mode 0 and 0 on the higher modes.
__global__ void boundary_dirichlet_kernel(const int* fcell, int64_t face0, int64_t nf, int nt, unsigned char* dmask,
                                          double* uD, double value) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nf * nt) return;
  const int64_t F = face0 + r / nt, R = face0 * nt + r;
  const bool b = fcell[2 * F + 1] < 0;
  dmask[R] = b ? 1 : 0;
  if (uD) uD[R] = (b && r % nt == 0) ? value : 0.0;
}

int blocks_for(int64_t n) { return (int)((n + 255) / 256 > 0 ? (n + 255) / 256 : 1); }

}  // namespace

int launch_rect_mesh(const RectMeshArgs& a, hipStream_t s) {
  const int64_t nn = (a.nx + 1) * (a.ny + 1);
  hipLaunchKernelGGL(rm_nodes_kernel, dim3(blocks_for(nn)), dim3(256), 0, s, a);
  hipLaunchKernelGGL(rm_cells_kernel, dim3(blocks_for(a.nx * a.ny)), dim3(256), 0, s, a);
  hipLaunchKernelGGL(rm_faces_kernel, dim3(blocks_for(a.nf)), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

int launch_boundary_dirichlet(const int* fcell, int64_t face0, int64_t nf, int nt, unsigned char* dmask, double* uD,
                              double value, hipStream_t s) {
  hipLaunchKernelGGL(boundary_dirichlet_kernel, dim3(blocks_for(nf * nt)), dim3(256), 0, s, fcell, face0, nf, nt,
                     dmask, uD, value);
  return (int)hipGetLastError();
}

}  // namespace hdg
