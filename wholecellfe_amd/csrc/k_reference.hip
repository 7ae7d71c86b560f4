// Kernels behind the reference-shaped stateless entry points (3 components
// per node, as the reference stores them) and the dense FP64 residual used by
// wcfe_dense_solve.
#include "wcfe_internal.hpp"

namespace wcfe {

// 6-knot force table of the kMD variant, UL_growth_explicit.cpp:1207-1214
// (extension in um, force in pN, stiffness in pN/um).
__constant__ double c_md_px[6] = {0., 2.51250583e-03, 4.40265201e-03, 5.91408228e-03, 11.76817302e-03, 17.001e-03};
__constant__ double c_md_py[6] = {-7.15514497, 71.80501308, 356.62420075, 356.96656556, 126.21811585, 528.40481124};
__constant__ double c_md_k[6] = {31426.8556, 99485.86235, 67080.67086, -7908.39043, 21978.66923, 76858.39733};

// UL:1258-1264: segment j for px_j <= D < px_{j+1}; D >= px_5 extrapolates the
// last segment.  D < 0 cannot occur (D is a norm).
__device__ __forceinline__ double md_force(double D) {
  int j = 0;
  if (D >= c_md_px[5]) {
    j = 5;
  } else {
    for (int q = 0; q < 5; ++q)
      if (D >= c_md_px[q] && D < c_md_px[q + 1]) j = q;
  }
  return c_md_py[j] + c_md_k[j] * (D - c_md_px[j]);
}

// calculateForce_FA (UL:1198-1303, law 1; UL1:1196-1295, law 0), one thread
// per node; the one-ring lists are in increasing triangle order.
__global__ __launch_bounds__(256) void k_ref_force_fa(int n_nodes, const int *ring_start, const int *ring,
                                                      const int *tris, const double *x, const double *cC,
                                                      const double *fau, int law, double kint, double *F) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_nodes) return;
  double Asum = 0.0;
  for (int k = ring_start[i]; k < ring_start[i + 1]; ++k) {
    const int *t = tris + 3 * ring[k];
    const double *p0 = x + 3 * t[0], *p1 = x + 3 * t[1], *p2 = x + 3 * t[2];
    const double e1[3] = {p1[0] - p0[0], p1[1] - p0[1], p1[2] - p0[2]};
    const double e2[3] = {p2[0] - p0[0], p2[1] - p0[1], p2[2] - p0[2]};
    const double nx = e1[1] * e2[2] - e1[2] * e2[1], ny = e1[2] * e2[0] - e1[0] * e2[2],
                 nz = e1[0] * e2[1] - e1[1] * e2[0];
    Asum += 0.5 * sqrt(nx * nx + ny * ny + nz * nz) / 3.0;
  }
  const double *u = fau + 3 * i;
  double fs[3];
  if (law == 0) {
    for (int c = 0; c < 3; ++c) fs[c] = kint * u[c];
  } else {
    const double D = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double f = md_force(D);
    for (int c = 0; c < 3; ++c) fs[c] = D == 0.0 ? 0.0 : f * (u[c] / D);
  }
  const double rho_i_max = 100.0;  // UL:1218
  for (int c = 0; c < 3; ++c) F[3 * i + c] = -cC[i] * fs[c] * Asum * rho_i_max;
}

void launch_ref_force_fa(hipStream_t s, int n_nodes, const int *ring_start, const int *ring, const int *tris,
                         const double *x, const double *cC, const double *fau, int law, double kint, double *F) {
  if (n_nodes <= 0) return;
  hipLaunchKernelGGL(k_ref_force_fa, dim3((n_nodes + 255) / 256), dim3(256), 0, s, n_nodes, ring_start, ring, tris, x,
                     cC, fau, law, kint, F);
}

// Point location on the substrate: the reference's containment test (signed
// z of two sub-triangle normals, A1 = A_tri - A2 - A3 >= 0; UL:2070-2095,
// UL:1335-1347) on the triangles of the point's cell of a uniform grid.  A
// cell lists every triangle whose (slightly widened) bounding box meets it,
// in increasing index, so scanning it visits every containing triangle in
// the reference's order.
__device__ __forceinline__ int grid_cell(const PointGrid &g, double px, double py) {
#pragma clang fp contract(off)
  const double fx = floor((px - g.ox) * g.inv_h), fy = floor((py - g.oy) * g.inv_h);
  const int ix = fx >= 0.0 ? (fx < g.gx ? (int)fx : g.gx - 1) : 0;  // NaN falls to cell 0 (no triangle contains it)
  const int iy = fy >= 0.0 ? (fy < g.gy ? (int)fy : g.gy - 1) : 0;
  return iy * g.gx + ix;
}
__device__ __forceinline__ bool tri_contains(const double *q0, const double *q1, const double *q2, const double *p,
                                             double &A_tri, double &A1, double &A2, double &A3) {
#pragma clang fp contract(off)
  const double e1[3] = {q1[0] - q0[0], q1[1] - q0[1], q1[2] - q0[2]};
  const double e2[3] = {q2[0] - q0[0], q2[1] - q0[1], q2[2] - q0[2]};
  const double ep[3] = {p[0] - q0[0], p[1] - q0[1], p[2] - q0[2]};
  const double nn[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
  A_tri = 0.5 * sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
  const double a3[3] = {e1[1] * ep[2] - e1[2] * ep[1], e1[2] * ep[0] - e1[0] * ep[2], e1[0] * ep[1] - e1[1] * ep[0]};
  A3 = -1.0;
  if (a3[2] >= 0.0) A3 = 0.5 * sqrt(a3[0] * a3[0] + a3[1] * a3[1] + a3[2] * a3[2]);
  const double a2[3] = {ep[1] * e2[2] - ep[2] * e2[1], ep[2] * e2[0] - ep[0] * e2[2], ep[0] * e2[1] - ep[1] * e2[0]};
  A2 = -1.0;
  if (a2[2] >= 0.0) A2 = 0.5 * sqrt(a2[0] * a2[0] + a2[1] * a2[1] + a2[2] * a2[2]);
  A1 = A_tri - A2 - A3;
  return A1 >= 0.0 && A2 >= 0.0 && A3 >= 0.0;
}

// One wave per node: its lanes test the candidate triangles of the node's grid
// cell at once (a chain of dependent loads per candidate: one thread per node
// walked them one after the other, 480 nodes 18 and 57 us; now 11 and 13, of
// which most is the launch and two cold memory round trips).
constexpr int POINT_WAVES = 4;  // nodes per workgroup

// updateFA 11-argument form (UL:2026-2174, law 1; UL1:2005-2115, law 0), one
// wave per cell node.  The substrate point X - fa_u is located among the
// substrate triangles (reference configuration) of its grid cell with the
// reference's z-sign tests; the last containing triangle wins (UL:2098).
__global__ __launch_bounds__(64 * POINT_WAVES) void k_ref_update_fa(int n_nodes, const double *X, const double *x,
                                                                    double *cA, double *cC, double *fau, double dt,
                                                                    PointGrid grid, const int *stris,
                                                                    const double *SX, const double *Sx, int law,
                                                                    double kint, int *n_unlocated) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * POINT_WAVES + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= n_nodes) return;
  double cell_u[3], sX[3], subs_u[3] = {0.0, 0.0, 0.0};
  for (int c = 0; c < 3; ++c) {
    cell_u[c] = x[3 * i + c] - X[3 * i + c];
    sX[c] = X[3 * i + c] - fau[3 * i + c];
  }
  bool located = false;
  const int gc = grid_cell(grid, sX[0], sX[1]);
  const int k1 = grid.start[gc + 1];
  for (int k0 = grid.start[gc]; k0 < k1; k0 += 64) {
    const int k = k0 + lane;
    bool in = false;
    double w[3] = {0.0, 0.0, 0.0};
    if (k < k1) {
      const int *t = stris + 3 * grid.list[k];
      double A_tri, A1, A2, A3;
      in = tri_contains(SX + 3 * t[0], SX + 3 * t[1], SX + 3 * t[2], sX, A_tri, A1, A2, A3);
      if (in)
        for (int c = 0; c < 3; ++c)
          w[c] = (A1 / A_tri) * (Sx[3 * t[0] + c] - SX[3 * t[0] + c]) +
                 (A2 / A_tri) * (Sx[3 * t[1] + c] - SX[3 * t[1] + c]) +
                 (A3 / A_tri) * (Sx[3 * t[2] + c] - SX[3 * t[2] + c]);
    }
    const unsigned long long hit = __ballot(in);
    if (hit) {  // last containing triangle wins (UL:2098)
      const int last = 63 - __clzll((long long)hit);
      for (int c = 0; c < 3; ++c) subs_u[c] = __shfl(w[c], last, 64);
      located = true;
    }
  }
  if (lane != 0) return;
  if (!located) atomicAdd(n_unlocated, 1);
  double u[3];
  for (int c = 0; c < 3; ++c) u[c] = fau[3 * i + c] + cell_u[c] - subs_u[c];
  double force;
  if (law == 0) {
    force = kint * sqrt(u[0] * u[0] + u[1] * u[1]);  // 2D norm, UL1:2077
  } else {
    const double D = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double f = md_force(D);
    double fs[3];
    for (int c = 0; c < 3; ++c) fs[c] = D == 0.0 ? 0.0 : f * (u[c] / D);
    force = sqrt(fs[0] * fs[0] + fs[1] * fs[1] + fs[2] * fs[2]);
  }
  const double k_on = 1.0, ka = 0.004, kb = 10.0, Fa = 15.0, Fb = 15.0;  // UL:2139-2143
  const double k_off = ka * shared_exp(force / Fa) + kb * shared_exp(-force / Fb);
  const double cold = cC[i];
  double cnew = cold + dt * k_on * (1.0 - cold) - dt * k_off * cold;
  if (cnew < 0.0) cnew = 0.0;
  if (cA[i] < 0.0) cA[i] = 0.0;
  cC[i] = cnew;
  const double keep = cold - dt * k_off * cold;
  for (int c = 0; c < 3; ++c) fau[3 * i + c] = (keep > 0.0 && cnew > 0.0) ? u[c] * keep / cnew : 0.0 * u[c];
}

void launch_ref_update_fa(hipStream_t s, int n_nodes, const double *X, const double *x, double *cA, double *cC,
                          double *fau, double dt, const PointGrid &grid, const int *stris, const double *SX,
                          const double *Sx, int law, double kint, int *n_unlocated) {
  if (n_nodes <= 0) return;
  hipLaunchKernelGGL(k_ref_update_fa, dim3((n_nodes + POINT_WAVES - 1) / POINT_WAVES), dim3(64 * POINT_WAVES), 0, s,
                     n_nodes, X, x, cA, cC, fau, dt,
                     grid, stris, SX, Sx, law, kint, n_unlocated);
}

// calculateForce_FA_subs (UL:1305-1475, law 1 MD table; UL1:1297, law 0
// linear kint), one wave per cell node: the node's integrin force at the
// substrate point x_cell - fa_u, for every substrate triangle containing it
// in the substrate's current positions, split by barycentric weight.  Each
// hit's 9 contributions are written out (hits in increasing triangle order,
// at most SUBS_MAX_HITS per node) and summed on the host in the reference's
// order.
__global__ __launch_bounds__(64 * POINT_WAVES) void k_ref_force_fa_subs(int n_nodes, const int *ring_start,
                                                                        const int *ring, const int *tris,
                                                                        const double *x_cell, const double *cC,
                                                                        const double *fau, PointGrid grid,
                                                                        const int *stris, const double *Sx, int law,
                                                                        double kint, SubsHits hits) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * POINT_WAVES + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= n_nodes) return;
  const double p[3] = {x_cell[3 * i] - fau[3 * i], x_cell[3 * i + 1] - fau[3 * i + 1],
                       x_cell[3 * i + 2] - fau[3 * i + 2]};
  const int gc = grid_cell(grid, p[0], p[1]);
  int h = 0;
  double Asum = -1.0, fs[3] = {0.0, 0.0, 0.0};
  const int k1 = grid.start[gc + 1];
  for (int k0 = grid.start[gc]; k0 < k1; k0 += 64) {
    const int k = k0 + lane;
    int e = 0;
    bool in = false;
    double A_tri = 1.0, A1 = 0.0, A2 = 0.0, A3 = 0.0;
    if (k < k1) {
      e = grid.list[k];
      const int *t = stris + 3 * e;
      in = tri_contains(Sx + 3 * t[0], Sx + 3 * t[1], Sx + 3 * t[2], p, A_tri, A1, A2, A3);
    }
    const unsigned long long hit = __ballot(in);
    if (!hit) continue;
    if (Asum < 0.0) {  // first hit: the node's one-ring area / 3 and its spring force
      Asum = 0.0;
      for (int r = ring_start[i]; r < ring_start[i + 1]; ++r) {
        const int *ct = tris + 3 * ring[r];
        const double *p0 = x_cell + 3 * ct[0], *p1 = x_cell + 3 * ct[1], *p2 = x_cell + 3 * ct[2];
        const double E1[3] = {p1[0] - p0[0], p1[1] - p0[1], p1[2] - p0[2]};
        const double E2[3] = {p2[0] - p0[0], p2[1] - p0[1], p2[2] - p0[2]};
        const double nx = E1[1] * E2[2] - E1[2] * E2[1], ny = E1[2] * E2[0] - E1[0] * E2[2],
                     nz = E1[0] * E2[1] - E1[1] * E2[0];
        Asum += 0.5 * sqrt(nx * nx + ny * ny + nz * nz) / 3;
      }
      const double *u = fau + 3 * i;
      if (law == 0) {
        for (int c = 0; c < 3; ++c) fs[c] = kint * u[c];
      } else {
        const double D = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
        const double f = md_force(D);
        for (int c = 0; c < 3; ++c) fs[c] = D == 0.0 ? 0.0 : f * (u[c] / D);
      }
    }
    const int at = h + __popcll(hit & ((1ull << lane) - 1ull));
    h += __popcll(hit);
    if (in && at < SUBS_MAX_HITS) {
      const bool near = at < SUBS_FIRST_HITS;
      const long long o = (long long)(near ? at : at - SUBS_FIRST_HITS) * n_nodes + i;
      (near ? hits.tri : hits.tri_more)[o] = e;
      double *v = (near ? hits.val : hits.val_more) + 9 * o;
      const double w[3] = {A1 / A_tri, A2 / A_tri, A3 / A_tri};
      const double rho_i_max = 100.0;  // UL:1391
      for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 3; ++c) v[3 * a + c] = cC[i] * fs[c] * w[a] * Asum * rho_i_max;
    }
    if (h > SUBS_MAX_HITS) break;
  }
  if (lane != 0) return;
  if (h > SUBS_MAX_HITS) atomicAdd(hits.overflow, 1);
  hits.n[i] = min(h, SUBS_MAX_HITS);
}
void launch_ref_force_fa_subs(hipStream_t s, int n_nodes, const int *ring_start, const int *ring, const int *tris,
                              const double *x_cell, const double *cC, const double *fau, const PointGrid &grid,
                              const int *stris, const double *Sx, int law, double kint, const SubsHits &hits) {
  if (n_nodes <= 0) return;
  hipLaunchKernelGGL(k_ref_force_fa_subs, dim3((n_nodes + POINT_WAVES - 1) / POINT_WAVES), dim3(64 * POINT_WAVES), 0, s,
                     n_nodes, ring_start, ring, tris, x_cell, cC, fau, grid, stris, Sx, law, kint, hits);
}

// The working-precision copy of the caller's matrices, one wave per row (24 systems
// of 60 to 700: 15 us; made on the host and sent as well it took 900).
template <class T>
__global__ __launch_bounds__(256) void k_dense_load(const CellParams *cp, const double *A64, const long long *a_off,
                                                    T *K) {
  const CellParams &p = cp[blockIdx.y];
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= p.npad) return;
  const double *A = A64 + a_off[blockIdx.y] + (long long)r * p.ndof;
  T *row = K + p.k_off + (long long)r * p.npad;
  for (int j = lane; j < p.npad; j += 64) row[j] = r < p.ndof && j < p.ndof ? (T)A[j] : (r == j ? T(1) : T(0));
}
template <class T>
void launch_dense_load(hipStream_t s, const CellParams *cp, int n_sys, int max_npad, const double *A64,
                       const long long *a_off, T *K) {
  if (n_sys <= 0 || max_npad <= 0) return;
  hipLaunchKernelGGL(k_dense_load<T>, dim3((max_npad + 3) / 4, n_sys), dim3(256), 0, s, cp, A64, a_off, K);
}
template void launch_dense_load<float>(hipStream_t, const CellParams *, int, int, const double *, const long long *,
                                       float *);
template void launch_dense_load<double>(hipStream_t, const CellParams *, int, int, const double *, const long long *,
                                        double *);

// r = b - A x in FP64 for dense systems; systems whose refinement has
// converged are skipped.  Bound by reading A once: one wave per row, its lanes
// along the row (512 contiguous bytes per load), RES_ROWS rows per workgroup
// so that every system spreads over the chip.  One thread per row in one
// workgroup per system read a different row in every lane: 179 us for 24
// systems of 60 to 700 unknowns.
constexpr int RES_ROWS = 16;
__global__ __launch_bounds__(256) void k_dense_residual(const CellParams *cp, const CellState *cs, const int *cells,
                                                        const double *A64, const long long *a_off, const double *b,
                                                        const double *x, double *r) {
  const int c = cells[blockIdx.y];
  if (cs[c].ir_done) return;
  const CellParams &p = cp[c];
  const int n = p.ndof, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double *A = A64 + a_off[c];
  const double *bb = b + p.vec_off, *xx = x + p.vec_off;
  double *rr = r + p.vec_off;
  const int i1 = min(n, ((int)blockIdx.x + 1) * RES_ROWS);
  for (int i = blockIdx.x * RES_ROWS + wave; i < i1; i += 4) {
    const double *row = A + (long long)i * n;
    double s0 = 0.0, s1 = 0.0;
    for (int j = lane; j < n; j += 128) {
      s0 += row[j] * xx[j];
      if (j + 64 < n) s1 += row[j + 64] * xx[j + 64];
    }
    s0 += s1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s0 += __shfl_xor(s0, o, 64);
    if (lane == 0) rr[i] = bb[i] - s0;
  }
}
void launch_dense_residual(hipStream_t s, const CellParams *cp, const CellState *cs, const int *cells, int ncell,
                           int max_ndof, const double *A64, const long long *a_off, const double *b, const double *x,
                           double *r) {
  if (ncell <= 0) return;
  hipLaunchKernelGGL(k_dense_residual, dim3((max_ndof + RES_ROWS - 1) / RES_ROWS, ncell), dim3(256), 0, s, cp, cs,
                     cells, A64, a_off, b, x, r);
}

// The shared FP64 exp over an array (diagnostics: bit-for-bit comparison with
// the same function compiled for the CPU).
__global__ __launch_bounds__(256) void k_eval_exp(long long n, const double *x, double *y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = shared_exp(x[i]);
}
void launch_eval_exp(hipStream_t s, long long n, const double *x, double *y) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_eval_exp, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, x, y);
}

}  // namespace wcfe
