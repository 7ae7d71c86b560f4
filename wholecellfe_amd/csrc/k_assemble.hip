// Assembly, FP64 residual/refinement vectors, Newton control and commit
// kernels for gfx950.
//
// Assembly is colour ordered: one launch per colour; within a colour no two
// elements share a node, so every += into the dense system and the residual
// has a single writer and the summation order per entry is fixed by the
// colour sequence (run-to-run bitwise deterministic, no atomics).
#include "cell_steps.hpp"

namespace wcfe {

// ---------------------------------------------------------------------------
// dense system fill: zero, identity on the padded diagonal (rows >= ndof)
// ---------------------------------------------------------------------------
template <class T> struct Vec16;
template <> struct Vec16<float> { typedef float4 type; static constexpr int n = 4; };
template <> struct Vec16<double> { typedef double2 type; static constexpr int n = 2; };

// lower_only: symmetric cells get the blocks (i, j) with j eliminated no later
// than i (rank) only: the band LU writes the others, U = L^T, before anything
// reads them
template <class T>
__global__ __launch_bounds__(256) void k_fill_systems(const CellParams *cp, const int *cells, int ncell, T *K,
                                                      const int *rank, int lower_only) {
  const int ci = blockIdx.y;
  if (ci >= ncell) return;
  const CellParams p = cp[cells[ci]];
  typedef typename Vec16<T>::type V;
  constexpr int VN = Vec16<T>::n;
  // blocks within the fill envelope |i - j| <= env only; a wave takes whole
  // 64-entry row segments, 64 * VN / 64 rows of a block at a time
  constexpr int LPR = 64 / VN;       // lanes per row segment
  constexpr int RPW = 64 / LPR;      // rows per wave
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane / LPR, lc = (lane % LPR) * VN;
  const bool lo = lower_only && p.sym;
  const int *rk = rank + p.rank_off;
  for (int r0 = RPW * (4 * (int)blockIdx.x + wave); r0 < p.npad; r0 += RPW * 4 * (int)gridDim.x) {
    const int rb = r0 / NB, r = r0 + lr;
    const int mine = lo ? rk[rb] : 0;
    T *row = K + p.k_off + (long long)r * p.npad;
    for (int jb = max(0, rb - p.env); jb <= min(p.nblk - 1, rb + p.env); ++jb) {
      if (lo && rk[jb] > mine) continue;
      T vals[VN];
#pragma unroll
      for (int k = 0; k < VN; ++k) vals[k] = (r >= p.ndof && r == jb * NB + lc + k) ? T(1) : T(0);
      V w;
      memcpy(&w, vals, sizeof(V));
      *reinterpret_cast<V *>(row + jb * NB + lc) = w;
    }
  }
}

template <class T>
void launch_fill_systems(hipStream_t s, const CellParams *cp, const int *cells, int ncell, int max_npad, T *K,
                         const int *rank, int lower_only) {
  if (ncell <= 0) return;
  // 16 (FP64: 8) rows per workgroup and pass; at most 64 workgroups per cell
  // of a large batch (the largest cells loop) so that small cells launch few
  // empty ones, and 2048 together of a small one (one cell of 20600 rows: 42 us
  // on 64 workgroups, 8 on 1284)
  const int rows = 4 * Vec16<T>::n;
  const int gx = std::max(1, std::min((max_npad + rows - 1) / rows, std::max(64, 2048 / ncell)));
  hipLaunchKernelGGL(k_fill_systems<T>, dim3(gx, ncell), dim3(256), 0, s, cp, cells, ncell, K, rank, lower_only);
}
template void launch_fill_systems<float>(hipStream_t, const CellParams *, const int *, int, int, float *, const int *,
                                         int);
template void launch_fill_systems<double>(hipStream_t, const CellParams *, const int *, int, int, double *,
                                          const int *, int);

__global__ __launch_bounds__(256) void k_fill(double *p, long long n, double value) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = value;
}
void launch_fill(hipStream_t s, double *p, long long n, double value) {
  if (n <= 0) return;
  long long b = (n + 255) / 256;
  int g = (int)(b < 4096 ? b : 4096);
  hipLaunchKernelGGL(k_fill, dim3(g), dim3(256), 0, s, p, n, value);
}

__global__ __launch_bounds__(256) void k_neg_copy(const double *src, double *dst, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dst[i] = -src[i];
}
void launch_neg_copy(hipStream_t s, const double *src, double *dst, long long n) {
  if (n <= 0) return;
  long long b = (n + 255) / 256;
  int g = (int)(b < 4096 ? b : 4096);
  hipLaunchKernelGGL(k_neg_copy, dim3(g), dim3(256), 0, s, src, dst, n);
}

// ---------------------------------------------------------------------------
// element assembly (one colour per launch)
// ---------------------------------------------------------------------------
template <class T, int MODE>
__global__ __launch_bounds__(128) void k_assemble(View v, int e_begin, int e_end, T *K, T *Kb, double *G,
                                                  double *Ke64, double *Rea, double *MM, CellState *cs) {
  const int e = e_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= e_end) return;
  const int c = v.el_cell[e];
  const int n[3] = {v.el_tri[3 * e], v.el_tri[3 * e + 1], v.el_tri[3 * e + 2]};
  if (MODE == ASM_STRAIN) {
    if (!v.cs[c].converged || v.cp[c].law != LAW_UL) return;
    double re[9], mm[3];
    element_strain(v, e, re, mm);
    for (int a = 0; a < 3; ++a) {
      for (int q = 0; q < 3; ++q) Rea[3 * n[a] + q] += re[3 * a + q];
      MM[n[a]] += mm[a];
    }
    return;
  }
  double Ge[6], Ke[36];
  bool ok = element_system<MODE == ASM_FULL>(v, e, Ge, Ke);
  if (!ok) cs[c].degenerate = 1;
  for (int a = 0; a < 3; ++a) {
    G[2 * n[a]] += Ge[2 * a];
    G[2 * n[a] + 1] += Ge[2 * a + 1];
  }
  if (MODE == ASM_FULL && v.cp[c].csr) {
    // block-CSR: the 3 x 3 node blocks of the element
    const int *bp = v.el_bpos + 9LL * e;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        T *B = Kb + 4LL * bp[3 * a + b];
        B[0] += T(Ke[(2 * a) * 6 + 2 * b]);
        B[1] += T(Ke[(2 * a) * 6 + 2 * b + 1]);
        B[2] += T(Ke[(2 * a + 1) * 6 + 2 * b]);
        B[3] += T(Ke[(2 * a + 1) * 6 + 2 * b + 1]);
      }
  } else if (MODE == ASM_FULL) {
    const CellParams &p = v.cp[c];
    T *A = K + p.k_off;
    const int kp[3] = {v.kpos[n[0]], v.kpos[n[1]], v.kpos[n[2]]};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int pp = 0; pp < 2; ++pp) {
        T *Ar = A + (long long)(2 * kp[a] + pp) * p.npad;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const int col = 2 * kp[b];
          Ar[col] += T(Ke[(2 * a + pp) * 6 + 2 * b]);
          Ar[col + 1] += T(Ke[(2 * a + pp) * 6 + 2 * b + 1]);
        }
      }
  }
  if (MODE == ASM_FULL && Ke64) {
    double2 *dst = reinterpret_cast<double2 *>(Ke64 + 36 * (long long)e);
#pragma unroll
    for (int k = 0; k < 18; ++k) dst[k] = make_double2(Ke[2 * k], Ke[2 * k + 1]);
  }
}

template <class T>
void launch_assemble(hipStream_t s, const View &v, int e_begin, int e_end, int mode, T *K, T *Kb, double *G,
                     double *Ke64, double *Rea, double *MM) {
  const int n = e_end - e_begin;
  if (n <= 0) return;
  dim3 grid((n + 127) / 128), block(128);
  CellState *cs = const_cast<CellState *>(v.cs);
  if (mode == ASM_FULL)
    hipLaunchKernelGGL((k_assemble<T, ASM_FULL>), grid, block, 0, s, v, e_begin, e_end, K, Kb, G, Ke64, Rea, MM,
                       cs);
  else if (mode == ASM_RESIDUAL)
    hipLaunchKernelGGL((k_assemble<T, ASM_RESIDUAL>), grid, block, 0, s, v, e_begin, e_end, K, Kb, G, Ke64, Rea, MM,
                       cs);
  else
    hipLaunchKernelGGL((k_assemble<T, ASM_STRAIN>), grid, block, 0, s, v, e_begin, e_end, K, Kb, G, Ke64, Rea, MM,
                       cs);
}
template void launch_assemble<float>(hipStream_t, const View &, int, int, int, float *, float *, double *, double *,
                                     double *, double *);
template void launch_assemble<double>(hipStream_t, const View &, int, int, int, double *, double *, double *,
                                      double *, double *, double *);

// ---------------------------------------------------------------------------
// whole-batch assembly in two launches: every element of every colour at once,
// then one thread per node gathering its rows.  A node's rows are written by
// that node's thread only, and it adds its elements' contributions in element
// order -- colour-major, the order the colour-by-colour scatter adds them -- so
// G and K are bit for bit the scatter's.
// ---------------------------------------------------------------------------
// FULL mode is bound by writing the element matrices (288 bytes each): a wave
// stages its 64 in LDS and stores them as one contiguous range (a store per
// thread and pair of entries, 288 bytes apart from lane to lane, reached
// 1.9 TB/s: 1.07 million elements 160 us, now 133).
constexpr int KE_PITCH = 37;  // doubles per element in LDS: lanes on different banks
template <int MODE>
__global__ __launch_bounds__(128) void k_element_pass(View v, int e_begin, int e_end, double *Ge_out, double *Ke64,
                                                      CellState *cs) {
  __shared__ double sh[MODE == ASM_FULL ? 2 * 64 * KE_PITCH : 1];
  const int e = e_begin + blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63, e0 = e - lane;
  double *ke = sh + (MODE == ASM_FULL ? (threadIdx.x >> 6) * 64 * KE_PITCH : 0);
  if (e < e_end) {
    double Ge[6], Ke[36];
    const bool ok = element_system<MODE == ASM_FULL>(v, e, Ge, Ke);
    if (!ok) cs[v.el_cell[e]].degenerate = 1;
    double2 *g = reinterpret_cast<double2 *>(Ge_out + 6LL * e);
#pragma unroll
    for (int k = 0; k < 3; ++k) g[k] = make_double2(Ge[2 * k], Ge[2 * k + 1]);
    if (MODE == ASM_FULL) {
#pragma unroll
      for (int k = 0; k < 36; ++k) ke[lane * KE_PITCH + k] = Ke[k];
    }
  }
  if (MODE == ASM_FULL) {
    __syncthreads();
    const int n = 18 * min(64, e_end - e0);  // pairs of the wave's elements (none: negative)
    double2 *dst = reinterpret_cast<double2 *>(Ke64 + 36LL * e0);
#pragma unroll
    for (int m = 0; m < 18; ++m) {
      const int j = lane + 64 * m;
      if (j < n) {
        const double *q = ke + (j / 18) * KE_PITCH + 2 * (j % 18);
        dst[j] = make_double2(q[0], q[1]);
      }
    }
  }
}

// RESIDUAL mode: each node gathers its two residual rows, element order
__global__ __launch_bounds__(256) void k_node_gather(const int *adj_start, const int *adj, int n0, int n1,
                                                     const double *Ge, double *G) {
  const int n = n0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= n1) return;
  double g0 = 0.0, g1 = 0.0;
  for (int k = adj_start[n]; k < adj_start[n + 1]; ++k) {
    const int pk = adj[k];
    const int e = pk >> 2, a = pk & 3;
    g0 += Ge[6LL * e + 2 * a];
    g1 += Ge[6LL * e + 2 * a + 1];
  }
  G[2 * n] = g0;
  G[2 * n + 1] = g1;
}

// FULL mode, one thread per group (row node n, column node): the 2 x 2
// block's contributions in element order, the order in which the
// colour-by-colour scatter adds them; the thread of the node's first group
// also gathers the node's residual rows.
template <class T>
__global__ __launch_bounds__(256) void k_group_gather(View v, const int *node_cell, const int *adj_start,
                                                      const int *adj, GatherPlan gp, const double *Ge,
                                                      const double *Ke64, double *G, T *K, T *Kb, int lower_only) {
  const int g = gp.g0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= gp.g1) return;
  const int n = gp.node[g];
  if (g == gp.start[n]) {
    double g0 = 0.0, g1 = 0.0;
    for (int k = adj_start[n]; k < adj_start[n + 1]; ++k) {
      const int pk = adj[k];
      const int e = pk >> 2, a = pk & 3;
      g0 += Ge[6LL * e + 2 * a];
      g1 += Ge[6LL * e + 2 * a + 1];
    }
    G[2 * n] = g0;
    G[2 * n + 1] = g1;
  }
  const int c = node_cell[n];
  const CellParams &p = v.cp[c];
  // lower_only: a symmetric cell's blocks whose column is eliminated after
  // their row are written by the fused band LU (U = L^T) before any read
  if (lower_only && p.sym && !p.csr) {
    const int *rk = v.rank + p.rank_off;
    if (rk[v.kpos[n] >> 5] < rk[v.kpos[gp.col[g]] >> 5]) return;
  }
  T *b0, *b1;
  if (p.csr) {
    if (gp.bpos[g] < 0) return;  // a node of no element
    b0 = Kb + 4LL * gp.bpos[g];
    b1 = b0 + 2;
  } else {
    b0 = K + p.k_off + 2LL * v.kpos[n] * p.npad + 2 * v.kpos[gp.col[g]];
    b1 = b0 + p.npad;
  }
  // the block's entries are zero (the fill or the sparse zero) before its one
  // group adds to them: no read.  The contributions four at a time, their
  // offsets and then their values loaded together, added in order.
  T a00 = T(0), a01 = T(0), a10 = T(0), a11 = T(0);
  const int q1 = gp.cstart[g + 1];
  for (int qb = gp.cstart[g]; qb < q1; qb += 4) {
    int o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) o[u] = qb + u < q1 ? gp.ke[qb + u] : -1;
    double2 x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (o[u] >= 0) {
        x[u] = *reinterpret_cast<const double2 *>(Ke64 + o[u]);
        y[u] = *reinterpret_cast<const double2 *>(Ke64 + o[u] + 6);
      }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (o[u] >= 0) {
        a00 += T(x[u].x);
        a01 += T(x[u].y);
        a10 += T(y[u].x);
        a11 += T(y[u].y);
      }
  }
  b0[0] = a00;
  b0[1] = a01;
  b1[0] = a10;
  b1[1] = a11;
}

template <class T>
void launch_assemble_gather(hipStream_t s, const View &v, int e_begin, int e_end, int mode, const int *node_cell,
                            const int *adj_start, const int *adj, const GatherPlan &gp, int n0, int n1, double *Ge,
                            double *Ke64, double *G, T *K, T *Kb, int lower_only) {
  CellState *cs = const_cast<CellState *>(v.cs);
  const int ne = e_end - e_begin, nn = n1 - n0;
  if (ne > 0) {
    if (mode == ASM_FULL)
      hipLaunchKernelGGL(k_element_pass<ASM_FULL>, dim3((ne + 127) / 128), dim3(128), 0, s, v, e_begin, e_end, Ge,
                         Ke64, cs);
    else
      hipLaunchKernelGGL(k_element_pass<ASM_RESIDUAL>, dim3((ne + 127) / 128), dim3(128), 0, s, v, e_begin, e_end,
                         Ge, Ke64, cs);
  }
  if (nn <= 0) return;
  const int ng = gp.g1 - gp.g0;
  if (mode == ASM_FULL) {
    if (ng > 0)
      hipLaunchKernelGGL((k_group_gather<T>), dim3((ng + 255) / 256), dim3(256), 0, s, v, node_cell, adj_start, adj,
                         gp, Ge, Ke64, G, K, Kb, lower_only);
  } else
    hipLaunchKernelGGL(k_node_gather, dim3((nn + 255) / 256), dim3(256), 0, s, adj_start, adj, n0, n1, Ge, G);
}
template void launch_assemble_gather<float>(hipStream_t, const View &, int, int, int, const int *, const int *,
                                            const int *, const GatherPlan &, int, int, double *, double *, double *,
                                            float *, float *, int);
template void launch_assemble_gather<double>(hipStream_t, const View &, int, int, int, const int *, const int *,
                                             const int *, const GatherPlan &, int, int, double *, double *, double *,
                                             double *, double *, int);

// One thread per node, each of its elements computed where it is needed: three
// times the (few) operations, but one launch and no intermediate arrays
// instead of two fills and a launch per colour.
__global__ __launch_bounds__(128) void k_node_strain(View v, const int *node_cell, const int *adj_start,
                                                     const int *adj, int n0, int n1, double *Rea, double *MM) {
  const int i = n0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n1) return;
  const int c = node_cell ? node_cell[i] : 0;
  if (!v.cs[c].converged || v.cp[c].law != LAW_UL) return;
  node_strain(v, i, adj_start, adj, Rea, MM);
}
void launch_node_strain(hipStream_t s, const View &v, const int *node_cell, const int *adj_start, const int *adj,
                        int n0, int n1, double *Rea, double *MM) {
  if (n1 <= n0) return;
  hipLaunchKernelGGL(k_node_strain, dim3((n1 - n0 + 127) / 128), dim3(128), 0, s, v, node_cell, adj_start, adj, n0, n1,
                     Rea, MM);
}

__global__ __launch_bounds__(128) void k_element_dump(View v, int e_begin, int e_end, double *Ge, double *Ke) {
  const int e = e_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= e_end) return;
  double g[6], k[36];
  element_system<true>(v, e, g, k);
  const long long o = e - e_begin;
  for (int i = 0; i < 6; ++i) Ge[6 * o + i] = g[i];
  for (int i = 0; i < 36; ++i) Ke[36 * o + i] = k[i];
}
void launch_element_dump(hipStream_t s, const View &v, int e_begin, int e_end, double *Ge, double *Ke) {
  const int n = e_end - e_begin;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_element_dump, dim3((n + 127) / 128), dim3(128), 0, s, v, e_begin, e_end, Ge, Ke);
}

// ---------------------------------------------------------------------------
// per-cell FP64 norms (fixed-order tree reduction, deterministic)
// which: 0 = residual after assembly (sets gnorm, bnorm and g0 at the first
//        iterate), 1 = refinement residual (rnorm), 2 = residual after the
//        update (gnorm)
// ---------------------------------------------------------------------------
// One workgroup per cell (blockIdx.x) and chunk (norm_chunks; blockIdx.y).  A cell of one chunk is summed by its one workgroup; a larger
// cell's chunks write partial sums and the last chunk to arrive adds them in
// chunk order (fixed order: bitwise reproducible).
// K (which 0, dense cells): also the factorization's pivot threshold from the
// diagonal.  Bound by latency: 16 waves, NORM_U entries of both in flight each
// (10300 nodes: 10 + 28 us as a norm and a threshold kernel of 4 waves, four
// entries in flight; now 7).
constexpr int NORM_THREADS = 1024, NORM_U = 8;
template <class T>
__global__ __launch_bounds__(NORM_THREADS) void k_cell_norm(const CellParams *cp, CellState *cs, const int *cells,
                                                            const double *vec, int which, int only_active,
                                                            double lin_rtol, NormWork nw, const T *K) {
  const int c = cells[blockIdx.x];
  const CellParams &p = cp[c];
  if (only_active && (cs[c].ir_done || p.refine)) return;
  const int nch = nw.part ? norm_chunks(p.ndof) : 1;
  const int per = (p.ndof + nch - 1) / nch;
  const int chunk = blockIdx.y;
  if (chunk >= nch) return;
  const double *v = vec + (long long)p.vec_off;
  const int lo = chunk * per, hi = min(p.ndof, lo + per);
  const bool tau = K && !p.csr;
  const T *A = K + p.k_off;
  double acc[NORM_U], m = 0.0;
#pragma unroll
  for (int u = 0; u < NORM_U; ++u) acc[u] = 0.0;
  for (int i0 = lo + threadIdx.x; i0 < hi; i0 += NORM_U * NORM_THREADS) {
    T d[NORM_U];
    double x[NORM_U];
#pragma unroll
    for (int u = 0; u < NORM_U; ++u) {
      const long long i = min(i0 + NORM_THREADS * u, hi - 1);
      x[u] = v[i];
      d[u] = tau ? A[i * p.npad + i] : T(0);
    }
#pragma unroll
    for (int u = 0; u < NORM_U; ++u) {
      if (i0 + NORM_THREADS * u < hi) acc[u] += x[u] * x[u];
      m = fmax(m, fabs((double)d[u]));  // fmax: a NaN is left out
    }
  }
#pragma unroll
  for (int w = NORM_U / 2; w > 0; w >>= 1)
#pragma unroll
    for (int u = 0; u < w; ++u) acc[u] += acc[u + w];
  __shared__ double red[NORM_THREADS], redm[NORM_THREADS];
  red[threadIdx.x] = acc[0];
  redm[threadIdx.x] = m;
  __syncthreads();
  for (int w = NORM_THREADS / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      red[threadIdx.x] += red[threadIdx.x + w];
      redm[threadIdx.x] = fmax(redm[threadIdx.x], redm[threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  const double eps = sizeof(T) == 4 ? 5.9604644775390625e-08 : 1.1102230246251565e-16;
  double sum = red[0];
  m = redm[0];
  if (nch > 1) {
    double *part = nw.part + 2LL * c * nw.stride;
    part[2 * chunk] = sum;
    part[2 * chunk + 1] = m;
    const unsigned prev = __hip_atomic_fetch_add(nw.cnt + c, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (prev != (unsigned)(nch - 1)) return;  // not the last chunk of the cell to arrive
    __hip_atomic_store(nw.cnt + c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sum = m = 0.0;
    for (int k = 0; k < nch; ++k) {
      sum += __hip_atomic_load(part + 2 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      m = fmax(m, __hip_atomic_load(part + 2 * k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
  }
  norm_finish(cs[c], which, sqrt(sum), lin_rtol);
  if (tau) tau_finish(cs[c], m, eps);
}
template <class T>
void launch_cell_norm(hipStream_t s, const CellParams *cp, CellState *cs, const int *cells, int ncell,
                      const double *vec, int which, int only_active, double lin_rtol, const NormWork &nw, const T *K) {
  if (ncell <= 0) return;
  const int nx = nw.part ? std::max(1, nw.stride) : 1;
  hipLaunchKernelGGL(k_cell_norm<T>, dim3(ncell, nx), dim3(NORM_THREADS), 0, s, cp, cs, cells, vec, which, only_active,
                     lin_rtol, nw, K);
}
template void launch_cell_norm<float>(hipStream_t, const CellParams *, CellState *, const int *, int, const double *,
                                      int, int, double, const NormWork &, const float *);
template void launch_cell_norm<double>(hipStream_t, const CellParams *, CellState *, const int *, int, const double *,
                                       int, int, double, const NormWork &, const double *);

// ---------------------------------------------------------------------------
// FP64 refinement residual r = -G - K d, element by element from the stored
// FP64 element matrices, gathered per node over its incident elements in
// element order (deterministic, no atomics)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_matvec_ir(const int *el_tri, const int *node_cell, const int *adj_start,
                                                   const int *adj, const double *Ke64, const double *G,
                                                   const double *delta, double *r, int node_begin, int node_end,
                                                   const CellState *cs, const CellParams *cp, BndView bv) {
  const int i = node_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= node_end) return;
  const int c = node_cell[i];
  if (cs[c].ir_done || cp[c].refine) return;
  const double2 ri = residual_node(i, el_tri, adj_start, adj, Ke64, G, delta, cp[c], bv, bv.gd ? bv.gd[c] : 0.0);
  r[2 * i] = ri.x;
  r[2 * i + 1] = ri.y;
}
void launch_matvec_ir(hipStream_t s, const View &v, const int *node_cell, const int *adj_start, const int *adj,
                      const double *Ke64, const double *G, const double *delta, double *r, int node_begin,
                      int node_end, const CellState *cs, const BndView &bv) {
  const int n = node_end - node_begin;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_matvec_ir, dim3((n + 255) / 256), dim3(256), 0, s, v.el_tri, node_cell, adj_start, adj, Ke64,
                     G, delta, r, node_begin, node_end, cs, v.cp, bv);
}

// Dense cells solve in their band-reducing numbering: rp = P r before the
// triangular solves, delta (+)= P^T dp after (cells still refining only).
__global__ __launch_bounds__(256) void k_perm_gather(const int *node_cell, const CellParams *cp, const int *kpos,
                                                     const double *r, double *rp, int n0, int n1) {
  const int n = n0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= n1) return;
  const CellParams &p = cp[node_cell[n]];
  if (p.csr) return;
  const long long o = 2LL * (p.node_off + kpos[n]);
  rp[o] = r[2LL * n];
  rp[o + 1] = r[2LL * n + 1];
}
__global__ __launch_bounds__(256) void k_perm_scatter(const int *node_cell, const CellParams *cp, const CellState *cs,
                                                      const int *kpos, const double *dp, double *delta, int n0, int n1,
                                                      int accumulate) {
  const int n = n0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= n1) return;
  const int c = node_cell[n];
  const CellParams &p = cp[c];
  if (p.csr || cs[c].ir_done) return;
  const long long o = 2LL * (p.node_off + kpos[n]);
  double *d = delta + 2LL * n;
  d[0] = accumulate ? d[0] + dp[o] : dp[o];
  d[1] = accumulate ? d[1] + dp[o + 1] : dp[o + 1];
}
void launch_perm_gather(hipStream_t s, const int *node_cell, const CellParams *cp, const int *kpos, const double *r,
                        double *rp, int n0, int n1) {
  if (n1 <= n0) return;
  hipLaunchKernelGGL(k_perm_gather, dim3((n1 - n0 + 255) / 256), dim3(256), 0, s, node_cell, cp, kpos, r, rp, n0, n1);
}
void launch_perm_scatter(hipStream_t s, const int *node_cell, const CellParams *cp, const CellState *cs,
                         const int *kpos, const double *dp, double *delta, int n0, int n1, int accumulate) {
  if (n1 <= n0) return;
  hipLaunchKernelGGL(k_perm_scatter, dim3((n1 - n0 + 255) / 256), dim3(256), 0, s, node_cell, cp, cs, kpos, dp, delta,
                     n0, n1, accumulate);
}

__global__ __launch_bounds__(256) void k_update_x(double2 *x, const double *delta, int node_begin, int node_end) {
  const int i = node_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= node_end) return;
  double2 p = x[i];
  p.x += delta[2 * i];
  p.y += delta[2 * i + 1];
  x[i] = p;
}
void launch_update_x(hipStream_t s, double2 *x, const double *delta, int node_begin, int node_end) {
  const int n = node_end - node_begin;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_update_x, dim3((n + 255) / 256), dim3(256), 0, s, x, delta, node_begin, node_end);
}

__global__ void k_newton_control(CellState *cs, const int *cells, int ncell, double rtol, double atol) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ncell) newton_finish(cs[cells[i]], rtol, atol);
}
void launch_newton_control(hipStream_t s, CellState *cs, const int *cells, int ncell, double rtol, double atol) {
  if (ncell <= 0) return;
  hipLaunchKernelGGL(k_newton_control, dim3((ncell + 63) / 64), dim3(64), 0, s, cs, cells, ncell, rtol, atol);
}

// ---------------------------------------------------------------------------
// commit of a converged load step
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_commit_nodes(View v, const int *node_cell, double2 *X, double2 *x, double *ea,
                                                      double *cC, double2 *fau, const double *Rea, const double *MM,
                                                      int node_begin, int node_end, double dt) {
  const int i = node_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= node_end) return;
  const int c = node_cell[i];
  if (!v.cs[c].converged) return;
  commit_node(v, v.cp[c], i, X, x, ea, cC, fau, Rea, MM, dt);
}
void launch_commit_nodes(hipStream_t s, const View &v, const int *node_cell, double2 *X, double2 *x, double *ea,
                         double *cC, double2 *fau, const double *Rea, const double *MM, int node_begin, int node_end,
                         double dt) {
  const int n = node_end - node_begin;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_commit_nodes, dim3((n + 255) / 256), dim3(256), 0, s, v, node_cell, X, x, ea, cC, fau, Rea, MM,
                     node_begin, node_end, dt);
}

__global__ __launch_bounds__(256) void k_commit_springs(View v, const int *sp_cell, const int *sp_elem,
                                                        const int *sp_local, double *state, double *anchor,
                                                        int s_begin, int s_end, BellArgs bell) {
  const int s = s_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= s_end) return;
  const int c = sp_cell[s];
  const CellState &cst = v.cs[c];
  if (!cst.converged) return;
  const CellParams &p = v.cp[c];
  if (p.kinetics != KIN_BELL) return;
  commit_spring(v, p, c, (unsigned)cst.step, s, sp_elem, sp_local, state, anchor, bell);
}
void launch_commit_springs(hipStream_t s, const View &v, const int *sp_cell, const int *sp_elem, const int *sp_local,
                           double *state, double *anchor, int s_begin, int s_end, const BellArgs &bell) {
  const int n = s_end - s_begin;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_commit_springs, dim3((n + 255) / 256), dim3(256), 0, s, v, sp_cell, sp_elem, sp_local, state,
                     anchor, s_begin, s_end, bell);
}

// A remeshed cell's nodes from its old nodes (the host's remeshing maps): new
// node i takes w_i old[src0_i] + (1 - w_i) old[src1_i] of the start-of-step
// and current positions, the strain, the bound fraction and the spring
// extension -- El Topo's midpoint interpolation of a split vertex
// (edgesplitter.cpp:563-577) is w = 1/2, a kept or renumbered vertex
// (defragmentation, surftrack.cpp:487-600) w = 1.  Rounded as written.
__global__ __launch_bounds__(256) void k_remap_nodes(int n_new, const int *src0, const int *src1, const double *w,
                                                     int old_off, const double2 *X, const double2 *x, const double *ea,
                                                     const double *cC, const double2 *fau, double2 *Xn, double2 *xn,
                                                     double *ean, double *cCn, double2 *faun) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_new) return;
  const int a = old_off + src0[i], b = old_off + src1[i];
  const double wa = w[i], wb = 1.0 - w[i];
  auto mix2 = [&](const double2 *v) { return make_double2(wa * v[a].x + wb * v[b].x, wa * v[a].y + wb * v[b].y); };
  Xn[i] = mix2(X);
  xn[i] = mix2(x);
  faun[i] = mix2(fau);
  cCn[i] = wa * cC[a] + wb * cC[b];
  for (int q = 0; q < 3; ++q) ean[3 * i + q] = wa * ea[3 * a + q] + wb * ea[3 * b + q];
}
void launch_remap_nodes(hipStream_t s, int n_new, const int *src0, const int *src1, const double *w, int old_off,
                        const double2 *X, const double2 *x, const double *ea, const double *cC, const double2 *fau,
                        double2 *Xn, double2 *xn, double *ean, double *cCn, double2 *faun) {
  if (n_new <= 0) return;
  hipLaunchKernelGGL(k_remap_nodes, dim3((n_new + 255) / 256), dim3(256), 0, s, n_new, src0, src1, w, old_off, X, x,
                     ea, cC, fau, Xn, xn, ean, cCn, faun);
}

__global__ void k_commit_cells(CellState *cs, const int *cells, int ncell, double dt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncell) return;
  CellState &s = cs[cells[i]];
  if (!s.converged) return;
  s.time += dt;
  s.step += 1;
  s.newton_it = 0;
}
void launch_commit_cells(hipStream_t s, CellState *cs, const int *cells, int ncell, double dt) {
  if (ncell <= 0) return;
  hipLaunchKernelGGL(k_commit_cells, dim3((ncell + 63) / 64), dim3(64), 0, s, cs, cells, ncell, dt);
}

// plain device copy, 16 bytes per thread per iteration (bandwidth probe and
// the known-size reference for the FETCH_SIZE / WRITE_SIZE counters)
__global__ __launch_bounds__(256) void k_copy(const float4 *src, float4 *dst, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
void launch_copy(hipStream_t s, const void *src, void *dst, long long bytes) {
  const long long n = bytes / 16;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_copy, dim3(4096), dim3(256), 0, s, static_cast<const float4 *>(src), static_cast<float4 *>(dst),
                     n);
}

}  // namespace wcfe
