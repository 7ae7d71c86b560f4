// 64 x 64 tiles on MFMA and in LDS, shared by the dense LU (k_lu.hip) and the
// band LU (k_band.hip).
#pragma once
#include <type_traits>
#include <utility>

#include "wcfe_internal.hpp"

namespace wcfe {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  Remap the workgroup id so that every XCD receives one contiguous
// range of work items: the tiles of one cell and block row then share an L2.
__device__ __forceinline__ int xcd_item(int b, int n) {
  const int q = n >> 3, r = n & 7, x = b & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// Dinv layout: per cell, per diagonal block k: L_kk^-1 (64 x 64 row-major,
// unit diagonal included) then U_kk^-1.
__device__ __forceinline__ long long dinv_off(const CellParams &p, int k) {
  return (long long)p.sys_off * 128 + (long long)k * 8192;
}

template <class T> struct Pitch { static constexpr int v = 68; };
template <> struct Pitch<double> { static constexpr int v = 66; };

// ---------------------------------------------------------------------------
// 64 x 64 x 64 products on MFMA.  4 waves, each a 32 x 32 quadrant = 2 x 2
// MFMA 16x16 tiles.  Operand layout of v_mfma_*_16x16x4: lane l supplies
// A[l%16][l/16] and B[l/16][l%16].  Accumulator register r of lane l holds
//   f32: D[4(l/16) + r][l%16]      f64: D[l/16 + 4r][l%16]
// (both measured on gfx950 with row/column-tagged operands).
// ---------------------------------------------------------------------------
__device__ __forceinline__ floatx4 mfma16(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ doublex4 mfma16(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int acc_row(float, int lk, int r) { return 4 * lk + r; }
__device__ __forceinline__ int acc_row(double, int lk, int r) { return lk + 4 * r; }
template <class T> struct Acc4;
template <> struct Acc4<float> { typedef floatx4 type; };
template <> struct Acc4<double> { typedef doublex4 type; };

// Software pipeline of the LDS-operand MFMA loops: the operands of k step
// kk + 4 are read while the MFMAs of step kk run (two register stages; the
// scheduling barriers keep the compiler from sinking the reads to their
// first use, which costs one LDS latency per step).  The MFMA sequence of
// every accumulator is unchanged.
#define WCFE_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

// acc += sign * X(64x64, LDS pitch PX) Y(64x64, LDS pitch PY) for this wave's quadrant
template <class T, int PX, int PY>
__device__ __forceinline__ void mma_64(const T *xs, const T *ys, typename Acc4<T>::type acc[2][2], T sign) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  T a[2][2], b[2][2];
  auto load = [&](int s, int kk) {
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) a[s][ti] = xs[(wr + ti * 16 + lr) * PX + kk + lk];
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) b[s][tj] = ys[(kk + lk) * PY + wc + tj * 16 + lr];
  };
  load(0, 0);
#pragma unroll
  for (int kk = 0; kk < 64; kk += 4) {
    const int s = (kk >> 2) & 1;
    if (kk + 4 < 64) load(s ^ 1, kk + 4);
    WCFE_SCHED_FENCE();
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      const T x = sign * a[s][ti];
#pragma unroll
      for (int tj = 0; tj < 2; ++tj) acc[ti][tj] = mfma16(x, b[s][tj], acc[ti][tj]);
    }
    WCFE_SCHED_FENCE();
  }
}

// ---------------------------------------------------------------------------
// Diagonal block: its inverse by Gauss-Jordan elimination without
// interchanges (pivots below tau replaced by +-tau), in 16 x 16 sub-blocks.
// Per sub-block step kb: wave 0 inverts the diagonal sub-block P in place
// (cross-lane reads), then on MFMA
//   row kb:       A_kb,j <- P^-1 A_kb,j                 (j != kb)
//   other rows i: A_i,j  <- A_i,j - A_i,kb A_kb,j  (j != kb),  A_i,kb <- -A_i,kb P^-1
// one wave per block row, so each row's old A_i,kb is read before it is
// replaced.  The block is taken as factored A_kk = I A_kk: the stored pair is
// Li = I (not stored when Li is null) and Ui = A_kk^-1, so the band LU's off-diagonal factors are
// L_ik = A_ik A_kk^-1 and U_kj = A_kj (block LDU form), and every solve that
// applies Li then Ui to a diagonal block applies A_kk^-1.
// a: the block in LDS (pitch PA), inverted in place; Li, Ui: 64 x 64
// row-major outputs (STORE).  All 256 threads call it (uniform barriers).
// Returns the pivots this thread replaced.
// ---------------------------------------------------------------------------
template <class T> __device__ __forceinline__ T rdlane(T v, int l);
template <> __device__ __forceinline__ float rdlane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
template <> __device__ __forceinline__ double rdlane(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __hiloint2double(hi, lo);
}

// reciprocal: the hardware's in FP32 (1 ulp, the factor is refined in FP64),
// IEEE division in FP64
__device__ __forceinline__ float recip(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ double recip(double v) { return 1.0 / v; }

// operand masks of the 16 x 16 products: as stored, unit lower, upper
enum : int { M_FULL = 0, M_UNIT_LOWER = 1, M_UPPER = 2 };
template <int M, class T> __device__ __forceinline__ T masked(T v, int r, int c) {
  if (M == M_UNIT_LOWER) return c < r ? v : (c == r ? T(1) : T(0));
  if (M == M_UPPER) return c >= r ? v : T(0);
  return v;
}

// acc += s X Y for 16 x 16 sub-blocks X, Y in LDS (pitch PA), one wave
template <class T, int PA, int MX, int MY>
__device__ __forceinline__ void mm16(const T *X, const T *Y, typename Acc4<T>::type &acc, T s) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  T xv[4], yv[4];  // every operand read before the four chained MFMAs
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    xv[q] = X[lr * PA + 4 * q + lk];
    yv[q] = Y[(4 * q + lk) * PA + lr];
  }
  WCFE_SCHED_FENCE();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const T x = masked<MX>(xv[q], lr, 4 * q + lk);
    const T y = masked<MY>(yv[q], 4 * q + lk, lr);
    acc = mfma16(s * x, y, acc);
  }
}
// acc[j] += s X Y_j for three 16 x 16 products with the same X (one wave):
// the three chains interleaved, every operand read first.  Each
// accumulator's MFMA sequence is mm16's.
template <class T, int PA>
__device__ __forceinline__ void mm16x3(const T *X, const T *Y0, const T *Y1, const T *Y2,
                                       typename Acc4<T>::type (&acc)[3], T s) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const T *Y[3] = {Y0, Y1, Y2};
  T xv[4], yv[3][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    xv[q] = X[lr * PA + 4 * q + lk];
#pragma unroll
    for (int j = 0; j < 3; ++j) yv[j][q] = Y[j][(4 * q + lk) * PA + lr];
  }
  WCFE_SCHED_FENCE();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const T x = s * xv[q];
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[j] = mfma16(x, yv[j][q], acc[j]);
  }
}
template <class T, int PA>
__device__ __forceinline__ void acc16_load(typename Acc4<T>::type &acc, const T *Z) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = Z[acc_row(T(0), lk, r) * PA + lr];
}
template <class T, int PA>
__device__ __forceinline__ void acc16_store(const typename Acc4<T>::type &acc, T *Z) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) Z[acc_row(T(0), lk, r) * PA + lr] = acc[r];
}

// 16 x 16 sub-block at D (pitch PA) inverted in place, one wave: lane l
// holds row l & 15, columns 4 (l >> 4) .. +3; the pivot and the pivot row and
// column reach the other lanes by cross-lane reads.
// FP32: the pivot row by DPP row broadcast (row_newbcast: lane j of each
// 16-lane row) and the pivot column by permlane32 / permlane16 swaps (row gj
// of the wave copied to all four rows): no LDS round trip on the chain.
template <int J> __device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + J, 0xF, 0xF, false));
}
template <int G> __device__ __forceinline__ float wave_row_bcast(float v) {
  const int x = __float_as_int(v);
  const auto h = __builtin_amdgcn_permlane32_swap(x, x, false, false);  // rows (0,1,0,1) | (2,3,2,3)
  const int y = G < 2 ? h[0] : h[1];
  const auto q = __builtin_amdgcn_permlane16_swap(y, y, false, false);  // even row | odd row, everywhere
  return __int_as_float(G % 2 == 0 ? q[0] : q[1]);
}
template <int J>
__device__ __forceinline__ void gj16_step(float (&v)[4], int lane, int r, int g, float tau, int &fixed) {
  constexpr int GJ = J >> 2, QJ = J & 3;
  const float p0 = rdlane(v[QJ], GJ * 16 + J);
  const bool small = !(fabsf(p0) >= tau);
  const float piv = small ? (p0 >= 0.0f ? tau : -tau) : p0;
  fixed += (small && lane == 0) ? 1 : 0;
  const float ip = recip(piv);
  const float f = wave_row_bcast<GJ>(v[QJ]);  // A[r][J]
  float rq[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) rq[q] = row_bcast<J>(v[q]) * ip;  // pivot row / pivot
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool cj = 4 * g + q == J;
    v[q] = (r == J) ? (cj ? ip : rq[q]) : (cj ? -f * ip : v[q] - f * rq[q]);
  }
}
template <int... J>
__device__ __forceinline__ void gj16_steps(float (&v)[4], int lane, int r, int g, float tau, int &fixed,
                                           std::integer_sequence<int, J...>) {
  (gj16_step<J>(v, lane, r, g, tau, fixed), ...);
}

template <class T, int PA> __device__ __forceinline__ int gj16(T *D, T tau) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  if constexpr (sizeof(T) == 4) {
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = D[r * PA + 4 * g + q];
    int fixed = 0;
    gj16_steps(v, lane, r, g, (float)tau, fixed, std::make_integer_sequence<int, 16>{});
#pragma unroll
    for (int q = 0; q < 4; ++q) D[r * PA + 4 * g + q] = v[q];
    return fixed;
  }
  T v[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = D[r * PA + 4 * g + q];
  int fixed = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int gj = j >> 2, qj = j & 3;
    const T p0 = rdlane(v[qj], gj * 16 + j);
    const bool small = !(fabs((double)p0) >= (double)tau);
    const T piv = small ? (p0 >= T(0) ? tau : -tau) : p0;
    fixed += (small && lane == 0) ? 1 : 0;
    const T ip = recip(piv);
    const T f = __shfl(v[qj], gj * 16 + r, 64);  // A[r][j]
    T rq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) rq[q] = __shfl(v[q], g * 16 + j, 64) * ip;  // pivot row / pivot
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool cj = 4 * g + q == j;
      v[q] = (r == j) ? (cj ? ip : rq[q]) : (cj ? -f * ip : v[q] - f * rq[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) D[r * PA + 4 * g + q] = v[q];
  return fixed;
}

template <class T, int PA, bool STORE>
__device__ __forceinline__ int invert_diag(T *a, T *Li, T *Ui, T tau) {
  typedef typename Acc4<T>::type acc_t;
  const int wave = threadIdx.x >> 6;
  int fixed = 0;
  auto sub = [](T *base, int i, int j) { return base + 16 * i * PA + 16 * j; };
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    if (wave == 0) fixed += gj16<T, PA>(sub(a, kb, kb), tau);
    __syncthreads();
    if (wave < 3) {  // row kb
      const int j = wave + (wave >= kb ? 1 : 0);
      acc_t acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = T(0);
      mm16<T, PA, M_FULL, M_FULL>(sub(a, kb, kb), sub(a, kb, j), acc, T(1));
      acc16_store<T, PA>(acc, sub(a, kb, j));
    }
    __syncthreads();
    if (wave < 3) {  // the other rows, one per wave
      const int i = wave + (wave >= kb ? 1 : 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j == kb) continue;
        acc_t acc;
        acc16_load<T, PA>(acc, sub(a, i, j));
        mm16<T, PA, M_FULL, M_FULL>(sub(a, i, kb), sub(a, kb, j), acc, T(-1));
        acc16_store<T, PA>(acc, sub(a, i, j));
      }
      acc_t acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = T(0);
      mm16<T, PA, M_FULL, M_FULL>(sub(a, i, kb), sub(a, kb, kb), acc, T(-1));
      acc16_store<T, PA>(acc, sub(a, i, kb));
    }
    __syncthreads();
  }
  if (STORE) {
    for (int idx = threadIdx.x; idx < 4096; idx += blockDim.x) {
      const int r = idx >> 6, c = idx & 63;
      if (Li) Li[idx] = r == c ? T(1) : T(0);
      Ui[idx] = a[r * PA + c];
    }
  }
  return fixed;
}

// invert_diag with work for the idle waves: wave 0 runs pre() and then the
// Gauss-Jordan inverse of sub-block kb while waves 1-3 run side(kb); every
// thread runs post(kb) right after that window's barrier.  The step's
// products take one phase (two barriers per sub-block step instead of
// three): with P the inverted pivot sub-block, wave 3 forms the new pivot
// row P A_kj in registers and stores it in the next window, while each other
// row's wave forms A'_ik = -A_ik P in place and then A_ij + A'_ik A_kj with
// the old pivot row -- the same elimination as invert_diag
// (A_ij - A_ik (P A_kj)), products associated the other way.
template <class T, int PA, bool STORE, class Pre, class Side, class Post>
__device__ __forceinline__ int invert_diag_ov(T *a, T *Li, T *Ui, T tau, Pre pre, Side side, Post post) {
  typedef typename Acc4<T>::type acc_t;
  const int wave = threadIdx.x >> 6;
  int fixed = 0;
  auto sub = [](T *base, int i, int j) { return base + 16 * i * PA + 16 * j; };
  acc_t rowk[3];  // wave 3: the new pivot row of the previous step
  auto store_row = [&](int kb) {
#pragma unroll
    for (int q = 0; q < 3; ++q) acc16_store<T, PA>(rowk[q], sub(a, kb, q + (q >= kb ? 1 : 0)));
  };
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    if (wave == 0) {
      if (kb == 0) pre();
      fixed += gj16<T, PA>(sub(a, kb, kb), tau);
    } else {
      if (wave == 3 && kb > 0) store_row(kb - 1);
      side(kb);
    }
    __syncthreads();
    post(kb);
    const int j0 = kb == 0 ? 1 : 0, j1 = kb <= 1 ? 2 : 1, j2 = kb <= 2 ? 3 : 2;  // the columns j != kb
    if (wave < 3) {  // row i: A'_ik = -A_ik P in place, then A_ij += A'_ik A_kj (old row kb)
      const int i = wave + (wave >= kb ? 1 : 0);
      acc_t o[3];
      acc16_load<T, PA>(o[0], sub(a, i, j0));
      acc16_load<T, PA>(o[1], sub(a, i, j1));
      acc16_load<T, PA>(o[2], sub(a, i, j2));
      acc_t acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = T(0);
      mm16<T, PA, M_FULL, M_FULL>(sub(a, i, kb), sub(a, kb, kb), acc, T(-1));
      acc16_store<T, PA>(acc, sub(a, i, kb));
      // the wave reads back what its lanes wrote: LDS operations of one
      // wave are performed in order; keep the compiler from reordering them
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      mm16x3<T, PA>(sub(a, i, kb), sub(a, kb, j0), sub(a, kb, j1), sub(a, kb, j2), o, T(1));
      acc16_store<T, PA>(o[0], sub(a, i, j0));
      acc16_store<T, PA>(o[1], sub(a, i, j1));
      acc16_store<T, PA>(o[2], sub(a, i, j2));
    } else {  // wave 3: the new row kb, P A_kj, kept until the next window
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) rowk[q][r] = T(0);
      mm16x3<T, PA>(sub(a, kb, kb), sub(a, kb, j0), sub(a, kb, j1), sub(a, kb, j2), rowk, T(1));
    }
    __syncthreads();
  }
  if (wave == 3) store_row(3);
  __syncthreads();
  if (STORE) {
    for (int idx = threadIdx.x; idx < 4096; idx += blockDim.x) {
      const int r = idx >> 6, c = idx & 63;
      if (Li) Li[idx] = r == c ? T(1) : T(0);
      Ui[idx] = a[r * PA + c];
    }
  }
  return fixed;
}

// A 64 x 64 tile in registers: each thread holds TileShape::E elements,
// moved as 16-byte vectors.
template <class T> struct TileShape {
  static constexpr int VN = 16 / sizeof(T);     // elements per vector
  static constexpr int PER_ROW = 64 / VN;       // vectors per row
  static constexpr int N = 64 * PER_ROW / 256;  // vectors per thread
  static constexpr int E = N * VN;              // elements per thread
};
template <class T>
__device__ __forceinline__ void tile_load(T (&t)[TileShape<T>::E], const T *g, long long ld) {
  typedef TileShape<T> R;
#pragma unroll
  for (int j = 0; j < R::N; ++j) {
    const int idx = threadIdx.x + 256 * j, r = idx / R::PER_ROW, c = (idx % R::PER_ROW) * R::VN;
    if constexpr (R::VN == 4) {
      const float4 v = *reinterpret_cast<const float4 *>(g + r * ld + c);
      t[4 * j] = v.x; t[4 * j + 1] = v.y; t[4 * j + 2] = v.z; t[4 * j + 3] = v.w;
    } else {
      const double2 v = *reinterpret_cast<const double2 *>(g + r * ld + c);
      t[2 * j] = v.x; t[2 * j + 1] = v.y;
    }
  }
}
template <class T, int P>
__device__ __forceinline__ void tile_to_lds(const T (&t)[TileShape<T>::E], T *s) {
  typedef TileShape<T> R;
#pragma unroll
  for (int j = 0; j < R::N; ++j) {
    const int idx = threadIdx.x + 256 * j, r = idx / R::PER_ROW, c = (idx % R::PER_ROW) * R::VN;
    if constexpr (R::VN == 4) {
      *reinterpret_cast<float4 *>(s + r * P + c) = make_float4(t[4 * j], t[4 * j + 1], t[4 * j + 2], t[4 * j + 3]);
    } else {
      *reinterpret_cast<double2 *>(s + r * P + c) = make_double2(t[2 * j], t[2 * j + 1]);
    }
  }
}

}  // namespace wcfe
