// Batched dense blocked LU for gfx950: right-looking, 64 x 64 blocks,
// row-major matrices padded to a multiple of 64 (identity on the padding).
//
// Every diagonal block k is factored once (L_kk \ U_kk stored in place) and
// the explicit inverses L_kk^-1, U_kk^-1 are kept in a side buffer (Dinv).
// That turns every block triangular solve of the factorisation into a
// 64 x 64 x 64 product on MFMA, and the diagonal solves of the triangular
// sweeps into small matrix-vector products.
//
// Per block step k, over every cell of the work list at once:
//   static pivoting, two block steps k, k+1 at a time (delayed update):
//                     [k = 0: k_lu_diag_inv]
//                     k_lu_trsm_mm   U_kj = L_kk^-1 A_kj, L_ik = A_ik U_kk^-1
//                     k_lu_gemm      strip: block column and row k+1 updated
//                                    with panel k only
//                     k_lu_trsm_mm   panel k+1
//                     k_lu_gemm      A_ij -= L_ik U_kj + L_i,k+1 U_k+1,j on
//                                    i, j >= k+2 (each C block read and
//                                    written once per two steps)
//                     The workgroup that finishes a diagonal block goes on
//                     to factor it and invert its triangles.
//                     Pivots below tau (64 eps max|K_ii|) are replaced by
//                     +-tau (static pivoting, Li & Demmel); FP64 iterative
//                     refinement removes the perturbation.
//   partial pivoting: k_lu_panel_pp  one workgroup factors the 64-wide
//                                    column panel with row interchanges
//                                    (LAPACK getf2 order inside the panel)
//                                    and inverts its diagonal triangles
//                     k_lu_laswp     interchanges on the trailing columns
//                                    only (LINPACK order)
//                     k_lu_trsm_mm   U_kj = L_kk^-1 A_kj
//                     k_lu_gemm
// MFMA: v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64.
// k_lu_solve applies the factors to one right-hand side per cell with the
// whole vector resident in LDS.
#include <hip/hip_ext.h>

#include "lu_tiles.hpp"

namespace wcfe {

// Work items: map[item] = (cell << 20) | index of the item within the cell.

// 64 x 64 block (row-major, leading dimension ld) <-> LDS tile with pitch P.
template <class T, int P>
__device__ __forceinline__ void load_block(T *s, const T *g, long long ld) {
  if (sizeof(T) == 4) {
    for (int idx = threadIdx.x; idx < 64 * 16; idx += blockDim.x) {
      const int r = idx >> 4, c = (idx & 15) * 4;
      const float4 v = *reinterpret_cast<const float4 *>(g + r * ld + c);
      *reinterpret_cast<float4 *>(s + r * P + c) = v;
    }
  } else {
    for (int idx = threadIdx.x; idx < 64 * 32; idx += blockDim.x) {
      const int r = idx >> 5, c = (idx & 31) * 2;
      const double2 v = *reinterpret_cast<const double2 *>(g + r * ld + c);
      *reinterpret_cast<double2 *>(s + r * P + c) = v;
    }
  }
}
template <class T, int P>
__device__ __forceinline__ void store_block(T *g, const T *s, long long ld) {
  if (sizeof(T) == 4) {
    for (int idx = threadIdx.x; idx < 64 * 16; idx += blockDim.x) {
      const int r = idx >> 4, c = (idx & 15) * 4;
      *reinterpret_cast<float4 *>(g + r * ld + c) = *reinterpret_cast<const float4 *>(s + r * P + c);
    }
  } else {
    for (int idx = threadIdx.x; idx < 64 * 32; idx += blockDim.x) {
      const int r = idx >> 5, c = (idx & 31) * 2;
      *reinterpret_cast<double2 *>(g + r * ld + c) = *reinterpret_cast<const double2 *>(s + r * P + c);
    }
  }
}

// Inverses of the unit lower and the upper triangle of the factored block in
// `a` (LDS), written row-major to Li and Ui (global).  Wave 0: column c of
// L^-1 by forward substitution; wave 1: column c of U^-1 by back substitution.
template <class T, int P>
__device__ __forceinline__ void invert_triangles(const T *a, T *Li, T *Ui) {
  const int w = threadIdx.x >> 6, c = threadIdx.x & 63;
  T x[64];
  if (w == 0) {
#pragma unroll
    for (int i = 0; i < 64; ++i) x[i] = (i == c) ? T(1) : T(0);
#pragma unroll
    for (int i = 1; i < 64; ++i) {
      T s = x[i];
#pragma unroll
      for (int m = 0; m < i; ++m) s -= a[i * P + m] * x[m];
      x[i] = s;
    }
#pragma unroll
    for (int i = 0; i < 64; ++i) Li[i * 64 + c] = x[i];
  } else if (w == 1) {
#pragma unroll
    for (int i = 63; i >= 0; --i) {
      T s = (i == c) ? T(1) : T(0);
#pragma unroll
      for (int m = i + 1; m < 64; ++m) s -= a[i * P + m] * x[m];
      x[i] = s / a[i * P + i];
    }
#pragma unroll
    for (int i = 0; i < 64; ++i) Ui[i * 64 + c] = x[i];
  }
}

// k = 0 of static pivoting: invert block (0, 0).
template <class T>
__global__ __launch_bounds__(256) void k_lu_diag_inv(const CellParams *cp, CellState *cs, const int *map, int k, T *K, T *Dinv) {
  constexpr int P = Pitch<T>::v;
  __shared__ T a[64 * P];
  const int v = map[blockIdx.x];
  const int c = v >> 20;
  const CellParams p = cp[c];
  const long long ld = p.npad;
  T *blk = K + p.k_off + (long long)(k * NB) * ld + k * NB;
  for (int idx = threadIdx.x; idx < 4096; idx += blockDim.x)
    a[(idx >> 6) * P + (idx & 63)] = blk[(idx >> 6) * ld + (idx & 63)];
  __syncthreads();
  T *D = Dinv + dinv_off(p, k);
  const int fixed = invert_diag<T, P, true>(a, D, D + 4096, (T)cs[c].tau);
  if (fixed) atomicAdd(&cs[c].n_static, fixed);
}
template <class T>
void launch_lu_diag_inv(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K,
                        T *Dinv) {
  if (wl.total <= 0) return;
  hipLaunchKernelGGL(k_lu_diag_inv<T>, dim3(wl.total), dim3(256), 0, s, cp, cs, wl.map, k, K,
                     Dinv);
}

// ---------------------------------------------------------------------------
// partial pivoting: panel factorisation (one workgroup per cell), then the
// inverses of the diagonal triangles
// ---------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(512) void k_lu_panel_pp(const CellParams *cp, CellState *cs, const int *map, int k, T *K, int *ipiv, T *Dinv) {
  constexpr int P = 65;
  __shared__ T prow[64];
  __shared__ double rv[16];
  __shared__ int ri[16];
  __shared__ int s_piv;
  __shared__ T a[64 * P];
  const int v = map[blockIdx.x];
  const int c = v >> 20;
  const CellParams p = cp[c];
  const long long ld = p.npad;
  T *A = K + p.k_off;
  int *piv_out = ipiv + p.sys_off;
  const int k0 = k * NB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int j = 0; j < 64; ++j) {
    const int col = k0 + j;
    double best = -1.0;
    int bi = 0x7fffffff;
    for (int r = col + threadIdx.x; r < p.npad; r += blockDim.x) {
      const double v = fabs((double)A[r * ld + col]);
      if (v > best) { best = v; bi = r; }
    }
    // wave argmax, ties to the lower row index
    for (int off = 32; off > 0; off >>= 1) {
      const double ov = __shfl_down(best, off, 64);
      const int oi = __shfl_down(bi, off, 64);
      if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
    }
    if (lane == 0) { rv[wave] = best; ri[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
      double b = rv[0];
      int i = ri[0];
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
        if (rv[w] > b || (rv[w] == b && ri[w] < i)) { b = rv[w]; i = ri[w]; }
      // a column of NaNs yields no candidate: keep the diagonal row
      if (i < col || i >= p.npad) i = col;
      s_piv = i;
      piv_out[col] = i;
      if (b == 0.0) cs[c].zero_pivot = 1;
    }
    __syncthreads();
    const int pr = s_piv;
    if (pr != col && threadIdx.x < 64) {
      const T t = A[col * ld + k0 + threadIdx.x];
      A[col * ld + k0 + threadIdx.x] = A[pr * ld + k0 + threadIdx.x];
      A[pr * ld + k0 + threadIdx.x] = t;
    }
    __syncthreads();
    if (threadIdx.x < 64) prow[threadIdx.x] = A[col * ld + k0 + threadIdx.x];
    __syncthreads();
    const T pv = prow[j];
    if (pv != T(0)) {
      for (int r = col + 1 + threadIdx.x; r < p.npad; r += blockDim.x) {
        T *row = A + r * ld + k0;
        const T l = row[j] / pv;
        row[j] = l;
        if (l != T(0))
          for (int cc = j + 1; cc < 64; ++cc) row[cc] -= l * prow[cc];
      }
    }
    __syncthreads();
  }
  T *blk = A + (long long)k0 * ld + k0;
  for (int idx = threadIdx.x; idx < 4096; idx += blockDim.x)
    a[(idx >> 6) * P + (idx & 63)] = blk[(idx >> 6) * ld + (idx & 63)];
  __syncthreads();
  T *D = Dinv + dinv_off(p, k);
  invert_triangles<T, P>(a, D, D + 4096);
}
// The same panel with its rows in registers: thread t owns rows k0 + t + 512 q
// (q < R), PSUB columns at a time.  What bounds it is the chain of 64 column
// steps, each a workgroup-wide argmax and the pivot row through LDS (two
// barriers); k_lu_panel_pp reads and writes every row's columns in global
// memory in each step.  A sub-panel takes the updates of the columns before it
// when it is loaded (its U rows by the first wave, which owns the panel's top
// 64 rows, then every row from LDS), and the interchanges of its columns reach
// the panel's other columns when it is done.  The pivot choice (largest
// magnitude, ties to the lower row) and every entry's operations and their
// order are k_lu_panel_pp's: the same pivots and factors.  Eight FP64 systems
// of 100 to 400 unknowns: 733 us per panel there; the whole solve 4.79 -> 1.96 ms
// with this form and the interchanges below.
constexpr int PANEL_THREADS = 512, PSUB = 16;

template <class T> struct Vec16B;
template <> struct Vec16B<float> { typedef float4 type; };
template <> struct Vec16B<double> { typedef double2 type; };
template <class T> __device__ __forceinline__ void row_load(T (&a)[PSUB], const T *g) {
  constexpr int VN = 16 / sizeof(T);
#pragma unroll
  for (int e = 0; e < PSUB; e += VN) {
    const typename Vec16B<T>::type v = *reinterpret_cast<const typename Vec16B<T>::type *>(g + e);
    __builtin_memcpy(&a[e], &v, sizeof v);
  }
}
template <class T> __device__ __forceinline__ void row_store(T *g, const T (&a)[PSUB]) {
  constexpr int VN = 16 / sizeof(T);
#pragma unroll
  for (int e = 0; e < PSUB; e += VN) {
    typename Vec16B<T>::type v;
    __builtin_memcpy(&v, &a[e], sizeof v);
    *reinterpret_cast<typename Vec16B<T>::type *>(g + e) = v;
  }
}

template <class T, int R>
__global__ __launch_bounds__(PANEL_THREADS) void k_lu_panel_reg(const CellParams *cp, CellState *cs, const int *map,
                                                                int k, T *K, int *ipiv, T *Dinv) {
  constexpr int P = 65, NWV = PANEL_THREADS / 64;
  __shared__ __attribute__((aligned(16))) T prow[2][PSUB], srow[2][PSUB], ub[2][PSUB][PSUB];
  __shared__ T rv[2][NWV], d[64 * P];
  __shared__ int ri[2][NWV], piv[64], zero[64], src[2 * PSUB], dst[2 * PSUB];
  const int c = map[blockIdx.x] >> 20;
  const CellParams p = cp[c];
  const long long ld = p.npad;
  T *A = K + p.k_off;
  const int k0 = k * NB, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T a[R][PSUB];
  for (int sp = 0; sp < 64 / PSUB; ++sp) {
    const int cb = k0 + sp * PSUB;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (k0 + tid + PANEL_THREADS * q < p.npad) row_load<T>(a[q], A + (k0 + tid + PANEL_THREADS * q) * ld + cb);
      else
#pragma unroll
        for (int e = 0; e < PSUB; ++e) a[q][e] = T(0);
    // the columns before this sub-panel, PSUB at a time
    for (int pb = 0; pb < sp; ++pb) {
      T(&u)[PSUB][PSUB] = ub[pb & 1];
      T l[R][PSUB];
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (k0 + tid + PANEL_THREADS * q < p.npad)
          row_load<T>(l[q], A + (k0 + tid + PANEL_THREADS * q) * ld + k0 + pb * PSUB);
        else
#pragma unroll
          for (int e = 0; e < PSUB; ++e) l[q][e] = T(0);
      if (wave == 0) {  // rows k0 .. k0 + 63: U rows top down, each once it is final
#pragma unroll
        for (int i = 0; i < PSUB; ++i) {
          if (lane == pb * PSUB + i) {
#pragma unroll
            for (int e = 0; e < PSUB; ++e) u[i][e] = a[0][e];
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          if (lane > pb * PSUB + i && l[0][i] != T(0) && !zero[pb * PSUB + i]) {
#pragma unroll
            for (int e = 0; e < PSUB; ++e) a[0][e] -= l[0][i] * u[i][e];
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < R; ++q) {
        if (wave == 0 && q == 0) continue;
#pragma unroll
        for (int i = 0; i < PSUB; ++i)
          if (l[q][i] != T(0) && !zero[pb * PSUB + i]) {
#pragma unroll
            for (int e = 0; e < PSUB; ++e) a[q][e] -= l[q][i] * u[i][e];
          }
      }
    }
#pragma unroll
    for (int J = 0; J < PSUB; ++J) {
      const int col = cb + J, o = J & 1;  // the row buffers alternate: a step's readers may lag behind the next writer
      T best = T(-1);
      int bi = 0x7fffffff;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int r = k0 + tid + PANEL_THREADS * q;
        const T v = a[q][J] < T(0) ? -a[q][J] : a[q][J];
        if (r >= col && r < p.npad && v > best) { best = v; bi = r; }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const T ov = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
      }
      if (lane == 0) { rv[o][wave] = best; ri[o][wave] = bi; }
      __syncthreads();
      T b = rv[o][0];
      int pr = ri[o][0];
#pragma unroll
      for (int w = 1; w < NWV; ++w) {
        const T ov = rv[o][w];
        const int oi = ri[o][w];
        if (ov > b || (ov == b && oi < pr)) { b = ov; pr = oi; }
      }
      if (pr < col || pr >= p.npad) pr = col;  // a column of NaNs yields no candidate: keep the diagonal row
      if (tid == 0) {
        piv[sp * PSUB + J] = pr;
        if (b == T(0)) cs[c].zero_pivot = 1;
      }
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int r = k0 + tid + PANEL_THREADS * q;
        if (r == pr) {
#pragma unroll
          for (int e = 0; e < PSUB; ++e) prow[o][e] = a[q][e];
        }
        if (r == col && pr != col) {
#pragma unroll
          for (int e = 0; e < PSUB; ++e) srow[o][e] = a[q][e];
        }
      }
      __syncthreads();
      const T pv = prow[o][J];
      if (tid == 0) zero[sp * PSUB + J] = pv == T(0);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int r = k0 + tid + PANEL_THREADS * q;
        if (pr != col) {  // the interchange
          if (r == col) {
#pragma unroll
            for (int e = 0; e < PSUB; ++e) a[q][e] = prow[o][e];
          }
          if (r == pr) {
#pragma unroll
            for (int e = 0; e < PSUB; ++e) a[q][e] = srow[o][e];
          }
        }
        if (pv != T(0) && r > col && r < p.npad) {
          const T l = a[q][J] / pv;
          a[q][J] = l;
          if (l != T(0)) {
#pragma unroll
            for (int e = J + 1; e < PSUB; ++e) a[q][e] -= l * prow[o][e];
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (k0 + tid + PANEL_THREADS * q < p.npad) row_store<T>(A + (k0 + tid + PANEL_THREADS * q) * ld + cb, a[q]);
    // this sub-panel's interchanges on the panel's other 48 columns: the
    // permutation they make (see k_lu_laswp), all reads before all writes
    if (tid < 2 * PSUB) {
      const int j = tid % PSUB, at = tid < PSUB ? cb + j : piv[sp * PSUB + j];
      int x = at;
      bool dup = false;
      for (int i = PSUB - 1; i >= 0; --i) {
        const int q = piv[sp * PSUB + i];
        if (x == cb + i) x = q;
        else if (x == q) x = cb + i;
        dup = dup || (i < j && q == at);
      }
      src[tid] = x;
      dst[tid] = (x == at || (tid >= PSUB && (at < cb + PSUB || dup))) ? -1 : at;
    }
    __syncthreads();
    {
      const int g = tid >> 4, e = tid & 15;  // position g, columns e, e + 16, e + 32 of the other 48
      T t[3];
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        const int cc = k0 + 16 * (w + (w >= sp ? 1 : 0)) + e;
        if (dst[g] >= 0) t[w] = A[src[g] * ld + cc];
      }
      __syncthreads();
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        const int cc = k0 + 16 * (w + (w >= sp ? 1 : 0)) + e;
        if (dst[g] >= 0) A[dst[g] * ld + cc] = t[w];
      }
    }
    __syncthreads();
  }
  if (tid < 64) ipiv[p.sys_off + k0 + tid] = piv[tid];
  const T *blk = A + (long long)k0 * ld + k0;
  for (int idx = tid; idx < 4096; idx += PANEL_THREADS) d[(idx >> 6) * P + (idx & 63)] = blk[(idx >> 6) * ld + (idx & 63)];
  __syncthreads();
  T *D = Dinv + dinv_off(p, k);
  invert_triangles<T, P>(d, D, D + 4096);
}
// rows: the most rows a panel of the list has left (npad - 64 k).  The
// register form holds R rows of PSUB entries (and their multipliers) per
// thread, up to 4 x 512 rows; longer panels stay in global memory.
template <class T>
void launch_lu_panel_pp(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K,
                        int *ipiv, T *Dinv, int rows) {
  if (wl.total <= 0) return;
  const dim3 g(wl.total), b(PANEL_THREADS);
  if (rows <= PANEL_THREADS)
    hipLaunchKernelGGL((k_lu_panel_reg<T, 1>), g, b, 0, s, cp, cs, wl.map, k, K, ipiv, Dinv);
  else if (rows <= 2 * PANEL_THREADS)
    hipLaunchKernelGGL((k_lu_panel_reg<T, 2>), g, b, 0, s, cp, cs, wl.map, k, K, ipiv, Dinv);
  else if (rows <= 4 * PANEL_THREADS)
    hipLaunchKernelGGL((k_lu_panel_reg<T, 4>), g, b, 0, s, cp, cs, wl.map, k, K, ipiv, Dinv);
  else
    hipLaunchKernelGGL(k_lu_panel_pp<T>, dim3(wl.total), dim3(512), 0, s, cp, cs, wl.map, k, K, ipiv, Dinv);
}

// Row interchanges of block k applied to the trailing columns [k0+64, npad).
// The 64 interchanges are one permutation of at most 128 rows: the rows k0 ..
// k0+63 and their pivot rows.  Lane j of the first wave follows position
// k0 + j backwards through the interchanges to the row whose content ends
// there, and likewise its pivot row's position; then every column's values
// are read, and after a barrier written: two dependent memory accesses
// instead of 64 (23.3 us per launch for 8 FP64 systems of 100 to 400).
template <class T>
__global__ __launch_bounds__(256) void k_lu_laswp(const CellParams *cp, const int *map,
                                                  int k, T *K, const int *ipiv) {
  __shared__ int pv[64], src[128], dst[128];
  const int v = map[blockIdx.x];
  const int c = v >> 20;
  const CellParams p = cp[c];
  const int chunk = v & 0xFFFFF;
  const int k0 = k * NB;
  if (threadIdx.x < 64) pv[threadIdx.x] = ipiv[p.sys_off + k0 + threadIdx.x];
  __syncthreads();
  if (threadIdx.x < 128) {
    const int j = threadIdx.x & 63;
    const int at = threadIdx.x < 64 ? k0 + j : pv[j];
    int x = at;
    bool dup = false;  // a pivot row inside the block, or named by an earlier interchange too
    for (int i = 63; i >= 0; --i) {
      const int q = pv[i];
      if (x == k0 + i) x = q;
      else if (x == q) x = k0 + i;
      dup = dup || (i < j && q == at);
    }
    src[threadIdx.x] = x;
    dst[threadIdx.x] = (x == at || (threadIdx.x >= 64 && (at < k0 + 64 || dup))) ? -1 : at;
  }
  __syncthreads();
  // 64 columns at a time, four threads per column, 32 rows each
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  T *A = K + p.k_off;
  const long long ld = p.npad;
  for (int cb = 0; cb < 4; ++cb) {
    const int col = k0 + NB + chunk * 256 + cb * 64 + lane;
    const bool ok = col < p.npad;
    T t[32];
#pragma unroll
    for (int u = 0; u < 32; ++u)
      if (ok && dst[4 * u + g] >= 0) t[u] = A[src[4 * u + g] * ld + col];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 32; ++u)
      if (ok && dst[4 * u + g] >= 0) A[dst[4 * u + g] * ld + col] = t[u];
  }
}
template <class T>
void launch_lu_laswp(hipStream_t s, const CellParams *cp, const WorkList &wl, int k, T *K, const int *ipiv) {
  if (wl.total <= 0) return;
  hipLaunchKernelGGL(k_lu_laswp<T>, dim3(wl.total), dim3(256), 0, s, cp, wl.map, k, K, ipiv);
}

// block triangular solves as products with the stored pair (Li, Ui):
//   items [0, m):  U_kj = Li_k A_kj
//   items [m, 2m): L_ik = A_ik Ui_k   (static pivoting only)
// Under static pivoting the pair is (I, A_kk^-1) (block LDU form, see
// invert_diag), so U_kj = A_kj and L_ik = A_ik A_kk^-1; under partial
// pivoting (U items only) Li_k is the inverse of the unit lower factor.
// Symmetric cells (p.sym) have only the L items, [0, m): U_ki = A_ik^T is
// stored by transposition of the block before the product.
template <class T>
__global__ __launch_bounds__(256) void k_lu_trsm_mm(const CellParams *cp, const int *map, int k, T *K,
                                                    const T *Dinv) {
  constexpr int P = Pitch<T>::v;
  typedef typename Acc4<T>::type acc_t;
  __shared__ __attribute__((aligned(16))) T xs[64 * P];
  __shared__ __attribute__((aligned(16))) T ys[64 * P];
  const int item = xcd_item(blockIdx.x, gridDim.x);
  const int v = map[item];
  const int c = v >> 20;
  const CellParams p = cp[c];
  const int t = v & 0xFFFFF;
  const int m = min(p.nblk - k - 1, p.bw);
  const bool upper = !p.sym && t < m;
  const int other = k + 1 + ((upper || p.sym) ? t : t - m);
  const long long ld = p.npad;
  T *A = K + p.k_off;
  const T *D = Dinv + dinv_off(p, k);
  T *blk = upper ? A + (long long)(k * NB) * ld + other * NB : A + (long long)(other * NB) * ld + k * NB;
  if (upper) {
    load_block<T, P>(xs, D, 64);
    load_block<T, P>(ys, blk, ld);
  } else {
    load_block<T, P>(xs, blk, ld);
    load_block<T, P>(ys, D + 4096, 64);
  }
  __syncthreads();
  acc_t acc[2][2];
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[ti][tj][r] = T(0);
  mma_64<T, P, P>(xs, ys, acc, T(1));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        blk[(long long)(wr + ti * 16 + acc_row(T(0), lk, r)) * ld + wc + tj * 16 + lr] = acc[ti][tj][r];
  if (!p.sym) return;
  // U_{k,other} = A_{other,k}^T, the block before the product (still in xs)
  T *U = A + (long long)(k * NB) * ld + other * NB;
  for (int idx = threadIdx.x; idx < 4096; idx += blockDim.x) {
    const int r = idx >> 6, cc = idx & 63;
    U[(long long)r * ld + cc] = xs[cc * P + r];
  }
}
template <class T>
void launch_lu_trsm(hipStream_t s, const CellParams *cp, CellState *, const WorkList &wl, int k, T *K,
                    const T *Dinv) {
  if (wl.total <= 0) return;
  hipLaunchKernelGGL(k_lu_trsm_mm<T>, dim3(wl.total), dim3(256), 0, s, cp, wl.map, k, K, Dinv);
}

// Trailing update C = A_ij - sum_p L_{i,k+p} U_{k+p,j} over np consecutive
// panels k .. k+np-1 (C is read and written once for np panels); the next
// panel's tiles are loaded into registers while the current one is on MFMA.
//   square mode: (i, j) over [s0, nblk)^2 with s0 = k + np (lower triangle
//                i >= j for symmetric cells)
//   strip mode:  target s0 = k + np: block column s0 from row s0 down, then
//                (non-symmetric cells) block row s0 from column s0 + 1 on --
//                the blocks panel s0 needs
// With `next_diag` (static pivoting) the workgroup of the diagonal block
// (s0, s0) then factors that block and stores the inverses of its triangles.
template <class T, bool STRIP>
__global__ __launch_bounds__(256) void k_lu_gemm(const CellParams *cp, CellState *cs, const int *map, int k, T *K,
                                                 T *Dinv, int next_diag, int np) {
  constexpr int P = Pitch<T>::v;
  typedef typename Acc4<T>::type acc_t;
  __shared__ __attribute__((aligned(16))) T ls[64 * P];
  __shared__ __attribute__((aligned(16))) T us[64 * P];
  const int item = xcd_item(blockIdx.x, gridDim.x);
  const int v = map[item];
  const int c = v >> 20;
  const CellParams p = cp[c];
  const int t = v & 0xFFFFF;
  const int s0 = k + np;
  int bi, bj;
  if (STRIP) {
    const int m = min(p.nblk - s0, p.bw);
    if (t < m) { bi = s0 + t; bj = s0; }
    else { bi = s0; bj = s0 + 1 + (t - m); }
  } else if (p.sym) {
    // lower triangle (i >= j) of the trailing matrix, row by row
    int i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (i * (i + 1) / 2 > t) --i;
    while ((i + 1) * (i + 2) / 2 <= t) ++i;
    bi = s0 + i;
    bj = s0 + (t - i * (i + 1) / 2);
  } else {
    const int mt = min(p.nblk - s0, p.bw);
    bi = s0 + t / mt;
    bj = s0 + t % mt;
  }
  T *A = K + p.k_off;
  const long long ld = p.npad;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  const int lk = lane >> 4, lr = lane & 15;
  T *C = A + (long long)(bi * NB) * ld + bj * NB;
  T lt[TileShape<T>::E], ut[TileShape<T>::E];
  tile_load<T>(lt, A + (long long)(bi * NB) * ld + k * NB, ld);
  tile_load<T>(ut, A + (long long)(k * NB) * ld + bj * NB, ld);
  acc_t acc[2][2];
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[ti][tj][r] = C[(long long)(wr + ti * 16 + acc_row(T(0), lk, r)) * ld + wc + tj * 16 + lr];
  for (int pn = 0; pn < np; ++pn) {
    if (pn) __syncthreads();  // the previous panel's products are done with the LDS tiles
    tile_to_lds<T, P>(lt, ls);
    tile_to_lds<T, P>(ut, us);
    __syncthreads();
    if (pn + 1 < np) {
      tile_load<T>(lt, A + (long long)(bi * NB) * ld + (k + pn + 1) * NB, ld);
      tile_load<T>(ut, A + (long long)((k + pn + 1) * NB) * ld + bj * NB, ld);
    }
    mma_64<T, P, P>(ls, us, acc, T(-1));
  }
  const bool diag_next = next_diag && bi == s0 && bj == s0;
  if (!diag_next) {
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
      for (int tj = 0; tj < 2; ++tj)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          C[(long long)(wr + ti * 16 + acc_row(T(0), lk, r)) * ld + wc + tj * 16 + lr] = acc[ti][tj][r];
    return;
  }
  // diagonal block s0 is final: factor it here
  __syncthreads();
  constexpr int PA = P;
  T *a = ls;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) a[(wr + ti * 16 + acc_row(T(0), lk, r)) * PA + wc + tj * 16 + lr] = acc[ti][tj][r];
  __syncthreads();
  T *D = Dinv + dinv_off(p, s0);
  const int fixed = invert_diag<T, PA, true>(a, D, D + 4096, (T)cs[c].tau);
  if (fixed) atomicAdd(&cs[c].n_static, fixed);
}
template <class T>
void launch_lu_gemm(hipStream_t s, const CellParams *cp, CellState *cs, const WorkList &wl, int k, T *K, T *Dinv,
                    int next_diag, int npanel, int strip, hipEvent_t ev_start, hipEvent_t ev_stop) {
  if (wl.total <= 0) return;
  if (ev_start) {  // profiling (never under graph capture): events at the kernel's own start and end
    if (strip)
      hipExtLaunchKernelGGL((k_lu_gemm<T, true>), dim3(wl.total), dim3(256), 0, s, ev_start, ev_stop, 0, cp, cs,
                            wl.map, k, K, Dinv, next_diag, npanel);
    else
      hipExtLaunchKernelGGL((k_lu_gemm<T, false>), dim3(wl.total), dim3(256), 0, s, ev_start, ev_stop, 0, cp, cs,
                            wl.map, k, K, Dinv, next_diag, npanel);
  } else if (strip) {
    hipLaunchKernelGGL((k_lu_gemm<T, true>), dim3(wl.total), dim3(256), 0, s, cp, cs, wl.map, k, K, Dinv, next_diag,
                       npanel);
  } else {
    hipLaunchKernelGGL((k_lu_gemm<T, false>), dim3(wl.total), dim3(256), 0, s, cp, cs, wl.map, k, K, Dinv, next_diag,
                       npanel);
  }
}

// ---------------------------------------------------------------------------
// triangular solves with the factors, one right-hand side per cell, the
// whole vector in LDS; diagonal blocks through the stored inverses
// ---------------------------------------------------------------------------
constexpr int SOLVE_THREADS = 512;

// y[k0 .. k0+63] <- Minv (64 x 64, row-major) * y[k0 .. k0+63]; 8 threads per row
template <class T>
__device__ __forceinline__ void diag_matvec(T *y, int k0, const T *Minv, T *tmp) {
  const int r = threadIdx.x >> 3, q = threadIdx.x & 7;
  T s = T(0);
  if (r < 64) {
    const T *row = Minv + r * 64 + q * 8;
#pragma unroll
    for (int c = 0; c < 8; ++c) s += row[c] * y[k0 + q * 8 + c];
  }
  s += __shfl_xor(s, 1, 64);
  s += __shfl_xor(s, 2, 64);
  s += __shfl_xor(s, 4, 64);
  if (r < 64 && q == 0) tmp[r] = s;
  __syncthreads();
  if (threadIdx.x < 64) y[k0 + threadIdx.x] = tmp[threadIdx.x];
  __syncthreads();
}

// y[rr] -= A[rr, k0 .. k0+63] . y[k0 .. k0+63] for rr in [r0, r1): a group of
// G lanes reads one row segment (G x 16 bytes, one coalesced 256 / 512-byte
// run), the partial dots are reduced across the group with shuffles.  Four
// rows per group are loaded before any arithmetic so the loads overlap.
template <class T>
__device__ __forceinline__ void block_column_update(T *y, const T *A, long long ld, int k0, int r0, int r1) {
  constexpr int V = 16 / sizeof(T);   // elements per 16-byte load
  constexpr int G = 64 / V;           // lanes per row segment
  constexpr int ROWS = SOLVE_THREADS / G;
  const int q = threadIdx.x % G, g = threadIdx.x / G;
  T yk[V];
#pragma unroll
  for (int e = 0; e < V; ++e) yk[e] = y[k0 + q * V + e];
  for (int base = r0; base < r1; base += 4 * ROWS) {
    T a[4][V];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int rr = base + u * ROWS + g;
      if (rr < r1) {
        const T *src = A + (long long)rr * ld + k0 + q * V;
        if constexpr (V == 4) {
          const float4 v = *reinterpret_cast<const float4 *>(src);
          a[u][0] = v.x; a[u][1] = v.y; a[u][2] = v.z; a[u][3] = v.w;
        } else {
          const double2 v = *reinterpret_cast<const double2 *>(src);
          a[u][0] = (T)v.x; a[u][1] = (T)v.y;
        }
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) a[u][e] = T(0);
      }
    }
    T sacc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      T t = T(0);
#pragma unroll
      for (int e = 0; e < V; ++e) t += a[u][e] * yk[e];
#pragma unroll
      for (int m = 1; m < G; m <<= 1) t += __shfl_xor(t, m, 64);
      sacc[u] = t;
    }
    if (q == 0)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int rr = base + u * ROWS + g;
        if (rr < r1) y[rr] -= sacc[u];
      }
  }
}

template <class T, bool PIVOT>
__global__ __launch_bounds__(SOLVE_THREADS) void k_lu_solve(const CellParams *cp, const CellState *cs,
                                                           const int *cells, const T *K, const T *Dinv,
                                                           const int *ipiv, const double *rhs, double *delta,
                                                           int accumulate) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ T tmp[64];
  T *y = reinterpret_cast<T *>(smem);
  const int c = cells[blockIdx.x];
  if (cs[c].ir_done) return;
  const CellParams p = cp[c];
  if (p.npad == 0) return;  // sparse cell: solved by PCG
  const T *A = K + p.k_off;
  const long long ld = p.npad;
  const double *r = rhs + (long long)p.vec_off;
  for (int i = threadIdx.x; i < p.npad; i += SOLVE_THREADS) y[i] = i < p.ndof ? (T)r[i] : T(0);
  __syncthreads();
  // forward: P, unit lower L (LINPACK order: block interchanges, then block)
  for (int kb = 0; kb < p.nblk; ++kb) {
    const int k0 = kb * NB;
    if (PIVOT) {
      if (threadIdx.x == 0) {
        const int *pv = ipiv + p.sys_off;
        for (int j = 0; j < 64; ++j) {
          const int q = pv[k0 + j];
          if (q != k0 + j) {
            const T tt = y[k0 + j];
            y[k0 + j] = y[q];
            y[q] = tt;
          }
        }
      }
      __syncthreads();
    }
    diag_matvec<T>(y, k0, Dinv + dinv_off(p, kb), tmp);
    block_column_update<T>(y, A, ld, k0, k0 + NB, min(p.npad, (kb + 1 + p.bw) * NB));  // rows in the band
    __syncthreads();
  }
  // backward: U with its diagonal
  for (int kb = p.nblk - 1; kb >= 0; --kb) {
    const int k0 = kb * NB;
    diag_matvec<T>(y, k0, Dinv + dinv_off(p, kb) + 4096, tmp);
    block_column_update<T>(y, A, ld, k0, max(0, (kb - p.bw) * NB), k0);
    __syncthreads();
  }
  double *dd = delta + (long long)p.vec_off;
  for (int i = threadIdx.x; i < p.ndof; i += SOLVE_THREADS) dd[i] = accumulate ? dd[i] + (double)y[i] : (double)y[i];
}

// ---------------------------------------------------------------------------
// Triangular solves for static pivoting across many workgroups: one workgroup
// per 64-row block row, every block row of every cell in one launch.
//   forward   y_k = L_kk^-1 (b_k - sum_{j<k} L_kj y_j)
//   backward  x_k = U_kk^-1 (y_k - sum_{j>k} U_kj x_j)      (x overwrites y)
// A workgroup streams its block row while the blocks it depends on are still
// being solved.  The solution entries are exchanged as self-validating 64-bit
// words (32-bit payload, 32-bit epoch; two words per FP64 entry) written and
// read with agent-scope atomics: a reader spins on the words it needs until
// they carry the current epoch, so no flag, fence or cache maintenance sits
// on the dependency chain.  The epoch advances by 2 per solve (forward E,
// backward E + 1), so stale words are never mistaken for new ones.
// Workgroups take their work item from a ticket counter, so every item a
// workgroup waits for belongs to a workgroup that started earlier; every wait
// is bounded (SPIN_LIMIT polls), after which the cell is flagged
// (CellState::solve_stall) and the workgroup finishes without waiting again.
// sync: [0] forward ticket, [1] backward ticket, [2] epoch, [3] any cell of
//       the list still refining (0: both sweeps return at once).
// ---------------------------------------------------------------------------
constexpr int MW_THREADS = 256;
constexpr int SPIN_LIMIT = 1 << 18;

__device__ __forceinline__ int mw_ticket(int *ticket, int *sh) {
  if (threadIdx.x == 0) *sh = atomicAdd(ticket, 1);
  __syncthreads();
  return *sh;
}

template <class T> struct MwShape {
  static constexpr int V = 16 / sizeof(T);  // elements per 16-byte load
  static constexpr int G = 64 / V;          // lanes per 64-element row segment
  static constexpr int RP = MW_THREADS / G; // rows per pass
  static constexpr int NP = 64 / RP;        // passes per 64-row block
  static constexpr int WPE = sizeof(T) / 4; // 64-bit words per exchanged entry
};

// part[u] += M[row_u, 0..63] . v[0..63] for this thread's slice, M a 64 x 64
// block (leading dimension ld), rows row_u = g + RP u, columns q V .. q V + V-1
template <class T>
__device__ __forceinline__ void mw_load_block(T (&a)[MwShape<T>::NP][MwShape<T>::V], const T *M, long long ld) {
  typedef MwShape<T> S;
  const int q = threadIdx.x % S::G, g = threadIdx.x / S::G;
#pragma unroll
  for (int u = 0; u < S::NP; ++u) {
    const T *src = M + (long long)(g + S::RP * u) * ld + q * S::V;
    if constexpr (S::V == 4) {
      const float4 v = *reinterpret_cast<const float4 *>(src);
      a[u][0] = v.x; a[u][1] = v.y; a[u][2] = v.z; a[u][3] = v.w;
    } else {
      const double2 v = *reinterpret_cast<const double2 *>(src);
      a[u][0] = v.x; a[u][1] = v.y;
    }
  }
}

template <class T>
__device__ __forceinline__ T mw_group_sum(T t) {
#pragma unroll
  for (int m = 1; m < MwShape<T>::G; m <<= 1) t += __shfl_xor(t, m, 64);
  return t;
}

__device__ __forceinline__ unsigned long long mw_word_load(const unsigned long long *w) {
  return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void mw_word_store(unsigned long long *w, unsigned payload, unsigned epoch) {
  __hip_atomic_store(w, ((unsigned long long)epoch << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Word w of the exchange buffer, already loaded into `v`: spin until it
// carries `epoch` (bounded).
__device__ __forceinline__ void mw_settle(unsigned long long &v, const unsigned long long *w, unsigned epoch,
                                          bool &gave_up, int *stall) {
  for (int spins = 0; (unsigned)(v >> 32) != epoch && !gave_up; ++spins) {
    if (spins >= SPIN_LIMIT) {
      gave_up = true;
      *stall = 1;
      break;
    }
    __builtin_amdgcn_s_sleep(2);
    v = mw_word_load(w);
  }
}

template <class T>
__device__ __forceinline__ T mw_decode(const unsigned long long *w) {
  if constexpr (MwShape<T>::WPE == 1) {
    return __uint_as_float((unsigned)w[0]);
  } else {
    return __hiloint2double((int)(unsigned)w[1], (int)(unsigned)w[0]);
  }
}

// Entry e of the exchange buffer, waiting until it carries `epoch`.
template <class T>
__device__ __forceinline__ T mw_get(const unsigned long long *yw, long long e, unsigned epoch, bool &gave_up,
                                    int *stall) {
  constexpr int WPE = MwShape<T>::WPE;
  unsigned long long w[WPE];
#pragma unroll
  for (int k = 0; k < WPE; ++k) w[k] = mw_word_load(yw + e * WPE + k);
#pragma unroll
  for (int k = 0; k < WPE; ++k) mw_settle(w[k], yw + e * WPE + k, epoch, gave_up, stall);
  return mw_decode<T>(w);
}

template <class T>
__device__ __forceinline__ void mw_put(unsigned long long *yw, long long e, T v, unsigned epoch) {
  if constexpr (MwShape<T>::WPE == 1) {
    mw_word_store(yw + e, __float_as_uint(v), epoch);
  } else {
    mw_word_store(yw + 2 * e, (unsigned)__double2loint(v), epoch);
    mw_word_store(yw + 2 * e + 1, (unsigned)__double2hiint(v), epoch);
  }
}

// One workgroup solves two consecutive block rows of the sweep: `rf`, then
// `rs` (rs = rf + 1 forward, rf - 1 backward; absent past the end), so the
// dependency chain has one cross-workgroup hop per two blocks.
template <class T>
__device__ __forceinline__ void mw_fetch_step(unsigned long long (&w)[MwShape<T>::V * MwShape<T>::WPE],
                                              const unsigned long long *ycw, int j, unsigned epoch, bool valid) {
  typedef MwShape<T> S;
  constexpr int NW = S::V * S::WPE;
  const int q = threadIdx.x % S::G;
  const long long base = (long long)j * NB * S::WPE + q * NW;
#pragma unroll
  for (int k = 0; k < NW; ++k) w[k] = valid ? mw_word_load(ycw + base + k) : ((unsigned long long)epoch << 32);
}

template <class T, bool FORWARD>
__global__ __launch_bounds__(MW_THREADS) void k_lu_solve_mw(const CellParams *cp, CellState *cs, const int *map,
                                                            const T *K, const T *Dinv, const double *rhs,
                                                            unsigned long long *yw, double *delta, const int *sync_c,
                                                            int *tickets, int accumulate) {
  typedef MwShape<T> S;
  constexpr int NW = S::V * S::WPE;
  constexpr int UNR = sizeof(T) == 4 ? 2 : 1;  // steps in flight per thread
  __shared__ int sh_ticket;
  __shared__ T vin[64];
  __shared__ T yf[64];
  if (sync_c[3] == 0) return;  // no cell of the list is refining
  const unsigned epoch_f = (unsigned)sync_c[2], epoch = epoch_f + (FORWARD ? 0u : 1u);
  const int item = map[mw_ticket(tickets + (FORWARD ? 0 : 1), &sh_ticket)];
  const int c = item >> 20, pi = item & 0xFFFFF;
  if (cs[c].ir_done) return;
  const CellParams p = cp[c];
  const long long ld = p.npad;
  // processing position of the first row; block of step s
  const int pf = 2 * pi;
  auto blk = [&](int st) { return FORWARD ? st : p.nblk - 1 - st; };
  const int rf = blk(pf);
  const bool two = pf + 1 < p.nblk;
  const int rs = two ? blk(pf + 1) : rf;
  const T *Af = K + p.k_off + (long long)(rf * NB) * ld;
  const T *As = K + p.k_off + (long long)(rs * NB) * ld;
  unsigned long long *ycw = yw + (long long)p.sys_off * S::WPE;
  int *stall = &cs[c].solve_stall;
  const int q = threadIdx.x % S::G, g = threadIdx.x / S::G;
  bool gave_up = false;
  // loaded before any wait: both diagonal inverses and the block (rs, rf)
  T dinf[S::NP][S::V], dins[S::NP][S::V], xs[S::NP][S::V];
  mw_load_block<T>(dinf, Dinv + dinv_off(p, rf) + (FORWARD ? 0 : 4096), 64);
  mw_load_block<T>(dins, Dinv + dinv_off(p, rs) + (FORWARD ? 0 : 4096), 64);
  mw_load_block<T>(xs, As + rf * NB, ld);
  T pf_[S::NP], ps_[S::NP];
#pragma unroll
  for (int u = 0; u < S::NP; ++u) pf_[u] = ps_[u] = T(0);
  // the blocks before rf within the band, in the order they are solved (the
  // first of them is one block beyond rs's band: zero in the fill envelope)
  for (int st = max(0, pf - p.bw); st < pf; st += UNR) {
    T a0[UNR][S::NP][S::V], a1[UNR][S::NP][S::V];
    unsigned long long w[UNR][NW];
#pragma unroll
    for (int i = 0; i < UNR; ++i) {
      const bool ok = st + i < pf;
      const int j = blk(ok ? st + i : st);
      if (ok) {
        mw_load_block<T>(a0[i], Af + j * NB, ld);
        if (two) mw_load_block<T>(a1[i], As + j * NB, ld);
      }
      mw_fetch_step<T>(w[i], ycw, j, epoch, ok);
    }
#pragma unroll
    for (int i = 0; i < UNR; ++i) {
      if (st + i >= pf) continue;
      const long long base = (long long)blk(st + i) * NB * S::WPE + q * NW;
#pragma unroll
      for (int k = 0; k < NW; ++k) mw_settle(w[i][k], ycw + base + k, epoch, gave_up, stall);
      T yv[S::V];
#pragma unroll
      for (int e = 0; e < S::V; ++e) yv[e] = mw_decode<T>(&w[i][e * S::WPE]);
#pragma unroll
      for (int u = 0; u < S::NP; ++u)
#pragma unroll
        for (int e = 0; e < S::V; ++e) {
          pf_[u] += a0[i][u][e] * yv[e];
          if (two) ps_[u] += a1[i][u][e] * yv[e];
        }
    }
  }
  // first row: y_rf = D_rf^-1 (b_rf - sum)
  const int k0f = rf * NB, k0s = rs * NB;
#pragma unroll
  for (int u = 0; u < S::NP; ++u) {
    const T sum = mw_group_sum<T>(pf_[u]);
    const int row = g + S::RP * u;
    if (q == 0) {
      T b;
      if (FORWARD) b = (k0f + row < p.ndof) ? (T)rhs[(long long)p.vec_off + k0f + row] : T(0);
      else b = mw_get<T>(ycw, k0f + row, epoch_f, gave_up, stall);
      vin[row] = b - sum;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < S::NP; ++u) {
    T t = T(0);
#pragma unroll
    for (int e = 0; e < S::V; ++e) t += dinf[u][e] * vin[q * S::V + e];
    t = mw_group_sum<T>(t);
    const int row = g + S::RP * u;
    if (q == 0) {
      mw_put<T>(ycw, k0f + row, t, epoch);
      yf[row] = t;
      if (!FORWARD && k0f + row < p.ndof) {
        double *dd = delta + (long long)p.vec_off + k0f + row;
        *dd = accumulate ? *dd + (double)t : (double)t;
      }
    }
  }
  if (!two) return;
  __syncthreads();
  // second row: y_rs = D_rs^-1 (b_rs - sum - A(rs, rf) y_rf)
#pragma unroll
  for (int u = 0; u < S::NP; ++u) {
#pragma unroll
    for (int e = 0; e < S::V; ++e) ps_[u] += xs[u][e] * yf[q * S::V + e];
    const T sum = mw_group_sum<T>(ps_[u]);
    const int row = g + S::RP * u;
    if (q == 0) {
      T b;
      if (FORWARD) b = (k0s + row < p.ndof) ? (T)rhs[(long long)p.vec_off + k0s + row] : T(0);
      else b = mw_get<T>(ycw, k0s + row, epoch_f, gave_up, stall);
      vin[row] = b - sum;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < S::NP; ++u) {
    T t = T(0);
#pragma unroll
    for (int e = 0; e < S::V; ++e) t += dins[u][e] * vin[q * S::V + e];
    t = mw_group_sum<T>(t);
    const int row = g + S::RP * u;
    if (q == 0) {
      mw_put<T>(ycw, k0s + row, t, epoch);
      if (!FORWARD && k0s + row < p.ndof) {
        double *dd = delta + (long long)p.vec_off + k0s + row;
        *dd = accumulate ? *dd + (double)t : (double)t;
      }
    }
  }
}

// Reset the tickets, advance the epoch and record whether any cell of the
// list is still refining (one workgroup).
__global__ __launch_bounds__(256) void k_solve_prepare(int *sync, const CellState *cs, const int *cells, int ncell) {
  __shared__ int any;
  if (threadIdx.x == 0) any = 0;
  __syncthreads();
  int a = 0;
  for (int i = threadIdx.x; i < ncell; i += 256) a |= cs[cells[i]].ir_done ? 0 : 1;
  if (a) any = 1;
  __syncthreads();
  if (threadIdx.x == 0) {
    sync[0] = 0;
    sync[1] = 0;
    sync[2] += 2;
    sync[3] = any;
  }
}

template <class T>
void launch_lu_solve_mw(hipStream_t s, const CellParams *cp, CellState *cs, const int *cells, int ncell,
                        const WorkList &fwd, const WorkList &bwd, const T *K, const T *Dinv, const double *r,
                        double *delta, void *yw, int *sync, int accumulate) {
  if (fwd.total <= 0) return;
  unsigned long long *w = static_cast<unsigned long long *>(yw);
  hipLaunchKernelGGL(k_solve_prepare, dim3(1), dim3(256), 0, s, sync, cs, cells, ncell);
  hipLaunchKernelGGL((k_lu_solve_mw<T, true>), dim3(fwd.total), dim3(MW_THREADS), 0, s, cp, cs, fwd.map, K, Dinv, r,
                     w, delta, sync, sync, accumulate);
  hipLaunchKernelGGL((k_lu_solve_mw<T, false>), dim3(bwd.total), dim3(MW_THREADS), 0, s, cp, cs, bwd.map, K, Dinv,
                     r, w, delta, sync, sync, accumulate);
}

size_t lu_solve_exchange_bytes(long long rows, int elem_size) { return (size_t)rows * 2 * elem_size; }

size_t lu_solve_lds_bytes(int npad, int elem_size) { return (size_t)npad * elem_size; }

// Dynamic LDS available to k_lu_solve next to its own static LDS.
size_t lu_solve_max_dynamic(size_t max_lds) { return max_lds > 1024 ? max_lds - 1024 : 0; }

hipError_t lu_prepare_attributes(size_t max_lds) {
  const int dyn = (int)lu_solve_max_dynamic(max_lds);
  const void *fns[] = {reinterpret_cast<const void *>(&k_lu_solve<float, true>),
                       reinterpret_cast<const void *>(&k_lu_solve<float, false>),
                       reinterpret_cast<const void *>(&k_lu_solve<double, true>),
                       reinterpret_cast<const void *>(&k_lu_solve<double, false>)};
  for (const void *f : fns) {
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
    if (e != hipSuccess) return e;
  }
  return band_prepare_attributes(max_lds);
}

template <class T>
void launch_lu_solve(hipStream_t s, const CellParams *cp, const CellState *cs, const int *cells, int ncell,
                     const T *K, const T *Dinv, const int *ipiv, int pivoting, const double *r, double *delta,
                     int max_npad, int accumulate) {
  if (ncell <= 0) return;
  const size_t lds = lu_solve_lds_bytes(max_npad, sizeof(T));
  if (pivoting)
    hipLaunchKernelGGL((k_lu_solve<T, true>), dim3(ncell), dim3(SOLVE_THREADS), lds, s, cp, cs, cells, K, Dinv, ipiv,
                       r, delta, accumulate);
  else
    hipLaunchKernelGGL((k_lu_solve<T, false>), dim3(ncell), dim3(SOLVE_THREADS), lds, s, cp, cs, cells, K, Dinv,
                       ipiv, r, delta, accumulate);
}

#define WCFE_INST(T)                                                                                                 \
  template void launch_lu_diag_inv<T>(hipStream_t, const CellParams *, CellState *, const WorkList &, int, T *, T *); \
  template void launch_lu_panel_pp<T>(hipStream_t, const CellParams *, CellState *, const WorkList &, int, T *,       \
                                      int *, T *, int);                                                               \
  template void launch_lu_laswp<T>(hipStream_t, const CellParams *, const WorkList &, int, T *, const int *);         \
  template void launch_lu_trsm<T>(hipStream_t, const CellParams *, CellState *, const WorkList &, int, T *,           \
                                  const T *);                                                                         \
  template void launch_lu_gemm<T>(hipStream_t, const CellParams *, CellState *, const WorkList &, int, T *, T *,      \
                                  int, int, int, hipEvent_t, hipEvent_t);                                             \
  template void launch_lu_solve<T>(hipStream_t, const CellParams *, const CellState *, const int *, int, const T *,   \
                                   const T *, const int *, int, const double *, double *, int, int);                  \
  template void launch_lu_solve_mw<T>(hipStream_t, const CellParams *, CellState *, const int *, int,               \
                                      const WorkList &, const WorkList &, const T *, const T *, const double *,      \
                                      double *, void *, int *, int);
WCFE_INST(float)
WCFE_INST(double)

}  // namespace wcfe
