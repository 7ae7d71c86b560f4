// Band LU of the dense cells (static pivoting): fused block steps and
// triangular sweeps over the plans of band_plan.hpp, for any number of leaves.
// FP32 (v_mfma_f32_16x16x4f32) and FP64 (v_mfma_f64_16x16x4f64).
#include <hip/hip_ext.h>

#include "cell_steps.hpp"
#include "lu_tiles.hpp"

namespace wcfe {

// The block step's B operand (the U tile) in LDS.  FP32: unpadded and
// swizzled, element (k, n) at 64 k + (n ^ 16 (k & 3)).  An MFMA B read takes
// rows kk .. kk+3 (lane group lk) and 16 consecutive columns (lr): the four
// row groups land on four different 16-bank groups, so the read is free of
// bank conflicts (a padded row pitch of 68 puts rows 4 words apart: up to
// four lanes on one bank).  FP64: the padded tile.  The same values in the
// same MFMA order.
template <class T> __device__ __forceinline__ int uidx(int k, int n) {
  if constexpr (sizeof(T) == 4) return 64 * k + (n ^ ((k & 3) << 4));
  else return Pitch<T>::v * k + n;
}
template <class T>
__device__ __forceinline__ void tile_to_lds_u(const T (&t)[TileShape<T>::E], T *s) {
  typedef TileShape<T> R;
#pragma unroll
  for (int j = 0; j < R::N; ++j) {
    const int idx = threadIdx.x + 256 * j, r = idx / R::PER_ROW, c = (idx % R::PER_ROW) * R::VN;
    if constexpr (R::VN == 4)
      *reinterpret_cast<float4 *>(s + uidx<T>(r, c)) = make_float4(t[4 * j], t[4 * j + 1], t[4 * j + 2], t[4 * j + 3]);
    else
      *reinterpret_cast<double2 *>(s + uidx<T>(r, c)) = make_double2(t[2 * j], t[2 * j + 1]);
  }
}
// acc += -X_I Y_J over k = 0..63 for the 16 x 16 output tile (I, J) of a
// 64 x 64 product, one wave; X in LDS (pitch P), Y a U tile.  The MFMA
// sequence per tile is mma_u's (same operands, same k order), so the tile
// comes out bit for bit as mma_u computes it.
template <class T, int P>
__device__ __forceinline__ void mmneg_tile_u(const T *X, const T *Y, int I, int J, typename Acc4<T>::type &acc) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < 64; kk += 4) {
    const T x = T(-1) * X[(I * 16 + lr) * P + kk + lk];
    const T y = Y[uidx<T>(kk + lk, J * 16 + lr)];
    acc = mfma16(x, y, acc);
  }
}
// The four tiles (I, 0..3) and the tile (0, J0) of the same product, one
// wave: each k step reads two X rows and four Y columns for five MFMAs on
// five independent accumulators (one tile at a time waits on its LDS reads
// every four MFMAs).  Each tile's MFMA sequence is mmneg_tile_u's.
template <class T, int P>
__device__ __forceinline__ void mmneg_row_u(const T *X, const T *Y, int I, int J0, typename Acc4<T>::type (&acc)[4],
                                            typename Acc4<T>::type &acc0) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll 4
  for (int kk = 0; kk < 64; kk += 4) {
    const T x = T(-1) * X[(I * 16 + lr) * P + kk + lk];
    const T x0 = T(-1) * X[lr * P + kk + lk];
    T y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = Y[uidx<T>(kk + lk, j * 16 + lr)];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = mfma16(x, y[j], acc[j]);
    acc0 = mfma16(x0, J0 == 1 ? y[1] : J0 == 2 ? y[2] : y[3], acc0);
  }
}
template <class T, int PX>
__device__ __forceinline__ void mma_u(const T *xs, const T *ys, typename Acc4<T>::type acc[2][2], T sign) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  T a[2][2], b[2][2];
  auto load = [&](int s, int kk) {
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) a[s][ti] = xs[(wr + ti * 16 + lr) * PX + kk + lk];
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) b[s][tj] = ys[uidx<T>(kk + lk, wc + tj * 16 + lr)];
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

// acc <- the 64 x 64 block at C (leading dimension ld), MFMA accumulator layout
template <class T>
__device__ __forceinline__ void acc_load64(typename Acc4<T>::type (&acc)[2][2], const T *C, long long ld, bool zero) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32, lk = lane >> 4, lr = lane & 15;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[ti][tj][r] = zero ? T(0) : C[(long long)(wr + ti * 16 + acc_row(T(0), lk, r)) * ld + wc + tj * 16 + lr];
}
template <class T>
__device__ __forceinline__ void acc_store64(const typename Acc4<T>::type (&acc)[2][2], T *C, long long ld) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32, lk = lane >> 4, lr = lane & 15;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) C[(long long)(wr + ti * 16 + acc_row(T(0), lk, r)) * ld + wc + tj * 16 + lr] = acc[ti][tj][r];
}
template <class T>
__device__ __forceinline__ void acc_zero(typename Acc4<T>::type (&acc)[2][2]) {
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[ti][tj][r] = T(0);
}
// the accumulator's block transposed to U (row-major, leading dimension ld):
// four consecutive entries of one row per lane
template <class T>
__device__ __forceinline__ void acc16_store_t(const typename Acc4<T>::type &acc, T *U, long long ld) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4 *>(U + (long long)lr * ld + 4 * lk) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) U[(long long)lr * ld + acc_row(T(0), lk, r)] = acc[r];
  }
}
template <class T>
__device__ __forceinline__ void acc_store64_t(const typename Acc4<T>::type (&acc)[2][2], T *U, long long ld) {
  const int w = threadIdx.x >> 6, wr = (w >> 1) * 32, wc = (w & 1) * 32;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) acc16_store_t<T>(acc[ti][tj], U + (long long)(wc + tj * 16) * ld + wr + ti * 16, ld);
}
template <class T, int P>
__device__ __forceinline__ void acc_to_lds(const typename Acc4<T>::type (&acc)[2][2], T *s) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32, lk = lane >> 4, lr = lane & 15;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < 2; ++tj)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[(wr + ti * 16 + acc_row(T(0), lk, r)) * P + wc + tj * 16 + lr] = acc[ti][tj][r];
}

__device__ __forceinline__ long long blk_off(int bi, int bj, long long ld) {
  return (long long)(bi * NB) * ld + (long long)(bj * NB);
}

// ---------------------------------------------------------------------------
// Fused block step: one launch per level of the plan.  In level l a pivot s
// takes the update of the pivot p of level l - 1 that reaches it, is inverted,
// and its column is solved (L_is = A_is A_ss^-1, and U_si = A_is^T for
// symmetric cells), while other items apply the pending updates of the other
// blocks.  What bounds a launch is the 64 x 64 inverse (four 16 x 16
// Gauss-Jordan steps, each a chain of 16 pivots): every INV item inverts
// block s from the same inputs, so no workgroup waits for another and only
// the STORE item's inverse is kept; diagonal blocks of K stay unfactored,
// nothing reads them afterwards.  How many column
// blocks an INV item takes and how many updated blocks another is chosen per
// launch by estimated time (LuPlan::choose_deal); the same products in the same
// order for every choice.
// ---------------------------------------------------------------------------

// forward substitution of the first solve (right-hand side -G in the band
// numbering), 4 lanes per row: the operations [f0, f0 + nf)
template <class T>
__device__ __forceinline__ void fwd_ops(const CellParams &p, const FwdOp *ops, int nf, const T *A, long long ld,
                                        StepFwd<T> fwd) {
  if (!fwd.y || nf == 0) return;
  T *y = fwd.y + p.sys_off;
  T *slots = fwd.slot + (long long)p.slot_off * NB;
  const int r = threadIdx.x >> 2, q = threadIdx.x & 3;
  T sum = T(0);
  for (int k = 0; k < nf; ++k) {
    const FwdOp o = ops[k];
    if (o.kind == FW_SUB) {
      if (q == 0) sum += slots[(long long)o.slot * NB + r];
      continue;
    }
    if (o.kind == FW_END) {
      if (q == 0) {
        const int i = o.i * NB + r, dof = fwd.kinv[p.sys_off + i];
        y[i] = (dof >= 0 ? (T)(-fwd.G[dof]) : T(0)) - sum;
      }
      sum = T(0);
      continue;
    }
    const T *Lr = A + blk_off(o.i, o.p, ld) + (long long)r * ld + q * 16;
    const T *yj = y + o.p * NB + q * 16;
    T part = T(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) part += Lr[e] * yj[e];
    part += __shfl_xor(part, 1, 64);
    part += __shfl_xor(part, 2, 64);
    if (q != 0) continue;
    if (o.kind == FW_TERM) {
      sum += part;
    } else {
      T *g = slots + (long long)o.slot * NB + r;
      *g = o.kind == FW_ACC0 ? part : *g + part;
    }
  }
}

// One item (see above).  All threads of the workgroup call it with the same
// arguments (uniform barriers); ls, us, xs are the workgroup's LDS tiles.
template <class T>
__device__ __forceinline__ void lu_step_item(const CellParams *cp, CellState *cs, const StepItem &it,
                                             const BlockRef *refs, const FwdOp *fops, T *K, T *Dinv, StepFwd<T> fwd,
                                             T *ls, T *us, T *xs) {
  constexpr int P = Pitch<T>::v, PA = P;
  typedef typename Acc4<T>::type acc_t;
  const CellParams &p = cp[it.cell];
  T *A = K + p.k_off;
  const long long ld = p.npad;
  const bool sym = p.sym != 0;
  refs += it.ref0;
  if (!(it.kind & STEP_INV)) {
    // the operand tiles of the next product are loaded while the current one
    // is on MFMA
    T lt[TileShape<T>::E], ut[TileShape<T>::E];
    auto operands = [&](const BlockRef &b, int pn) {
      tile_load<T>(lt, A + blk_off(b.bi, pn, ld), ld);
      tile_load<T>(ut, A + blk_off(pn, b.bj, ld), ld);
    };
    BlockRef b = it.nref > 0 ? refs[0] : BlockRef{0, 0, -1, -1, 1, 0};
    acc_t acc[2][2], nacc[2][2];
    if (it.nref > 0) {
      operands(b, b.p0);
      acc_load64<T>(acc, A + blk_off(b.bi, b.bj, ld), ld, b.first != 0);
    }
    for (int q = 0; q < it.nref; ++q) {
      const bool more = q + 1 < it.nref;
      const BlockRef next = more ? refs[q + 1] : b;
      if (q) __syncthreads();  // the previous block's products are done with ls / us
      tile_to_lds<T, P>(lt, ls);
      tile_to_lds_u<T>(ut, us);
      if (b.p1 >= 0) operands(b, b.p1);
      else if (more) operands(next, next.p0);
      if (more) acc_load64<T>(nacc, A + blk_off(next.bi, next.bj, ld), ld, next.first != 0);
      __syncthreads();
      mma_u<T, P>(ls, us, acc, T(-1));
      if (b.p1 >= 0) {
        __syncthreads();
        tile_to_lds<T, P>(lt, ls);
        tile_to_lds_u<T>(ut, us);
        if (more) operands(next, next.p0);
        __syncthreads();
        mma_u<T, P>(ls, us, acc, T(-1));
      }
      acc_store64<T>(acc, A + blk_off(b.bi, b.bj, ld), ld);
#pragma unroll
      for (int ti = 0; ti < 2; ++ti)
#pragma unroll
        for (int tj = 0; tj < 2; ++tj) acc[ti][tj] = nacc[ti][tj];
      b = next;
    }
    fwd_ops<T>(p, fops + it.fop0, it.nfop, A, ld, fwd);
    return;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lk = lane >> 4, lr = lane & 15;
  const int s = it.s, k = it.p;
  const bool store = (it.kind & STEP_STORE) != 0, own = it.nref > 0;
  const BlockRef r0 = own ? refs[0] : BlockRef{0, 0, -1, -1, 1, 0};
  T *C = A + blk_off(r0.bi, s, ld);
  T *D = Dinv + dinv_off(p, s) + 4096;  // the identity before it (L's diagonal) only where something reads it
  const T tau = (T)cs[it.cell].tau;
  acc_t acc[2][2];
  T *inv;  // the inverse's LDS tile, and the tile that stages a column block
  T *stage;
  T lt[TileShape<T>::E];
  acc_t pf[2][2];
  const bool two = it.nref >= 2;
  const BlockRef r1 = two ? refs[1] : BlockRef{0, 0, -1, -1, 1, 0};
  if (k >= 0) {
    // Pivot k updates block s (and the own block): the updates run inside the
    // inverse.  Block s -= L_sk U_ks: wave 0 takes sub-block (0,0) just
    // before its Gauss-Jordan step, waves 1-3 the other 15 meanwhile.  The
    // own block's 16 sub-blocks live in waves 1-3's registers; they take the
    // update A -= L_ik U_ks during steps 1-3 and are staged in ls for the
    // final product.  LDS: xs block s (then its inverse), ls L_sk (then L_ik,
    // then the own block), us U_ks.  Every tile's MFMA sequence is mma_u's.
    const bool upd_own = own && r0.p0 >= 0;
    T ld2[TileShape<T>::E], ut[TileShape<T>::E];
    tile_load<T>(lt, A + blk_off(s, s, ld), ld);
    tile_load<T>(ld2, A + blk_off(s, k, ld), ld);
    tile_load<T>(ut, A + blk_off(k, s, ld), ld);
    acc_t ow[6];
    if (own && w > 0) {
#pragma unroll
      for (int sl = 0; sl < 6; ++sl) {
        const int tt = (w - 1) + 3 * sl;
        if (tt < 16) {
          const T *Ct = C + (long long)((tt >> 2) * 16) * ld + (tt & 3) * 16;
#pragma unroll
          for (int r = 0; r < 4; ++r) ow[sl][r] = r0.first ? T(0) : Ct[(long long)acc_row(T(0), lk, r) * ld + lr];
        }
      }
    }
    tile_to_lds<T, P>(lt, xs);
    tile_to_lds<T, P>(ld2, ls);
    tile_to_lds_u<T>(ut, us);
    if (upd_own) tile_load<T>(lt, A + blk_off(r0.bi, k, ld), ld);
    // the second column block (and its L block of column k, below in post)
    // are loaded while the inverse runs
    if (two) acc_load64<T>(pf, A + blk_off(r1.bi, s, ld), ld, r1.first != 0);
    __syncthreads();
    auto pre = [&]() {
      acc_t d;
      acc16_load<T, PA>(d, xs);
      mmneg_tile_u<T, P>(ls, us, 0, 0, d);
      acc16_store<T, PA>(d, xs);
    };
    T *Ut = A + blk_off(s, r0.bi, ld);  // U_si (symmetric cells)
    auto side = [&](int kb) {
      if (kb == 0) {  // wave w: row w of the sub-blocks and sub-block (0, w)
        acc_t d[4], d0;
#pragma unroll
        for (int J = 0; J < 4; ++J) acc16_load<T, PA>(d[J], xs + w * 16 * PA + J * 16);
        acc16_load<T, PA>(d0, xs + w * 16);
        mmneg_row_u<T, P>(ls, us, w, w, d, d0);
#pragma unroll
        for (int J = 0; J < 4; ++J) acc16_store<T, PA>(d[J], xs + w * 16 * PA + J * 16);
        acc16_store<T, PA>(d0, xs + w * 16);
        return;
      }
      if (!own) return;
#pragma unroll
      for (int sl = 2 * (kb - 1); sl < 2 * kb; ++sl) {
        const int tt = (w - 1) + 3 * sl;
        if (tt >= 16) continue;
        const int I = tt >> 2, J = tt & 3;
        if (upd_own) mmneg_tile_u<T, P>(ls, us, I, J, ow[sl]);
        if (sym) acc16_store_t<T>(ow[sl], Ut + (long long)(J * 16) * ld + I * 16, ld);
      }
    };
    auto post = [&](int kb) {
      if (kb == 0 && upd_own) tile_to_lds<T, P>(lt, ls);  // L_sk is done with
      if (kb == 0 && two && r1.p0 >= 0) tile_load<T>(lt, A + blk_off(r1.bi, k, ld), ld);
      if (kb == 3 && own && w > 0) {
#pragma unroll
        for (int sl = 0; sl < 6; ++sl) {
          const int tt = (w - 1) + 3 * sl;
          if (tt < 16) acc16_store<T, P>(ow[sl], ls + (tt >> 2) * 16 * P + (tt & 3) * 16);
        }
      }
    };
    if (store) {
      const int fixed = invert_diag_ov<T, PA, true>(xs, fwd.store_id ? D - 4096 : nullptr, D, tau, pre, side, post);
      if (fixed) atomicAdd(&cs[it.cell].n_static, fixed);
    } else {
      (void)invert_diag_ov<T, PA, false>(xs, nullptr, D, tau, pre, side, post);
    }
    inv = xs;
    stage = ls;
  } else {
    // no pending update: block s and the own block as they are, the own block
    // staged in xs; U_si stored now (its stores overlap the inverse)
    acc_load64<T>(pf, A + blk_off(s, s, ld), ld, false);
    if (own) {
      acc_load64<T>(acc, C, ld, r0.first != 0);
      acc_to_lds<T, P>(acc, xs);
      if (sym) acc_store64_t<T>(acc, A + blk_off(s, r0.bi, ld), ld);
    }
    acc_to_lds<T, PA>(pf, us);
    if (two) acc_load64<T>(pf, A + blk_off(r1.bi, s, ld), ld, r1.first != 0);
    __syncthreads();
    if (store) {
      const int fixed = invert_diag<T, PA, true>(us, fwd.store_id ? D - 4096 : nullptr, D, tau);
      if (fixed) atomicAdd(&cs[it.cell].n_static, fixed);
    } else {
      (void)invert_diag<T, PA, false>(us, nullptr, D, tau);
    }
    inv = us;
    stage = xs;
  }
  if (!own) return;
  // the column's blocks, each as an item of its own computes it (same products
  // in the same order); pf and lt hold the next block and its L block of
  // column k, loaded while the current one is on MFMA
  for (int q = 0;; ++q) {
    const BlockRef b = q == 0 ? r0 : refs[q];
    const bool more = q + 1 < it.nref;
    if (q) {
      // stage is free (the barrier below); with a pending update it is ls, and us holds U_ks
      if (b.p0 >= 0) {
        tile_to_lds<T, P>(lt, stage);
        __syncthreads();
        mma_u<T, P>(stage, us, pf, T(-1));
        __syncthreads();
      }
      if (sym) acc_store64_t<T>(pf, A + blk_off(s, b.bi, ld), ld);
      acc_to_lds<T, P>(pf, stage);
      if (more) {
        const BlockRef n = refs[q + 1];
        acc_load64<T>(pf, A + blk_off(n.bi, s, ld), ld, n.first != 0);
        if (n.p0 >= 0) tile_load<T>(lt, A + blk_off(n.bi, k, ld), ld);
      }
      __syncthreads();
    }
    acc_zero<T>(acc);
    mma_64<T, P, PA>(stage, inv, acc, T(1));
    acc_store64<T>(acc, A + blk_off(b.bi, s, ld), ld);
    if (!more) return;
    __syncthreads();  // this block's product is done with the stage tile
  }
}

// LDS of a block step: three 64 x Pitch tiles (FP64: over the static limit)
template <class T> constexpr int step_lds() { return 3 * 64 * Pitch<T>::v * (int)sizeof(T); }

template <class T>
__device__ __forceinline__ void lu_step_body(const CellParams *cp, CellState *cs, const StepItem *items,
                                             const BlockRef *refs, const FwdOp *fops, T *K, T *Dinv, StepFwd<T> fwd,
                                             T *lds) {
  const StepItem it = items[xcd_item(blockIdx.x, gridDim.x)];
  lu_step_item<T>(cp, cs, it, refs, fops, K, Dinv, fwd, lds, lds + 64 * Pitch<T>::v, lds + 128 * Pitch<T>::v);
}
// One launch per level: every item of every cell in it.  FP32: 183 registers,
// two workgroups per compute unit; held to three (168 registers, 104 spilled)
// the 1,024-replica kind of batch is 2 % slower and the others the same.
// FP64: one workgroup per compute unit by its LDS.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_lu_step_f32(
    const CellParams *cp, CellState *cs, const StepItem *items, const BlockRef *refs, const FwdOp *fops, float *K,
    float *Dinv, StepFwd<float> fwd) {
  __shared__ __attribute__((aligned(16))) float lds[3 * 64 * Pitch<float>::v];
  lu_step_body<float>(cp, cs, items, refs, fops, K, Dinv, fwd, lds);
}
__global__ __launch_bounds__(256) void k_lu_step_f64(const CellParams *cp, CellState *cs, const StepItem *items,
                                                     const BlockRef *refs, const FwdOp *fops, double *K, double *Dinv,
                                                     StepFwd<double> fwd) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  lu_step_body<double>(cp, cs, items, refs, fops, K, Dinv, fwd, reinterpret_cast<double *>(smem));
}

// The whole factorization of a cell in one workgroup: its items in level
// order (panel form), a barrier between them.  The items of one level are
// independent (they run concurrently above), so any order inside a level
// gives the same results.  ranges: items [x, y) per cell, longest first.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_lu_cell_f32(
    const CellParams *cp, CellState *cs, const int2 *ranges, const StepItem *items, const BlockRef *refs,
    const FwdOp *fops, float *K, float *Dinv, StepFwd<float> fwd) {
  __shared__ __attribute__((aligned(16))) float lds[3 * 64 * Pitch<float>::v];
  const int2 rg = ranges[xcd_item(blockIdx.x, gridDim.x)];
  for (int i = rg.x; i < rg.y; ++i) {
    const StepItem it = items[i];
    lu_step_item<float>(cp, cs, it, refs, fops, K, Dinv, fwd, lds, lds + 64 * Pitch<float>::v,
                        lds + 128 * Pitch<float>::v);
    __syncthreads();  // the item's global writes are visible to the next item
  }
}

template <class T>
void launch_lu_step(hipStream_t s, const CellParams *cp, CellState *cs, const StepItem *items, int n,
                    const BlockRef *refs, const FwdOp *fops, T *K, T *Dinv, StepFwd<T> fwd, hipEvent_t ev_start,
                    hipEvent_t ev_stop) {
  if (n <= 0) return;
  if constexpr (sizeof(T) == 4) {
    if (ev_start)  // profiling (never under graph capture): events at the kernel's own start and end
      hipExtLaunchKernelGGL(k_lu_step_f32, dim3(n), dim3(256), 0, s, ev_start, ev_stop, 0, cp, cs, items, refs, fops,
                            K, Dinv, fwd);
    else
      hipLaunchKernelGGL(k_lu_step_f32, dim3(n), dim3(256), 0, s, cp, cs, items, refs, fops, K, Dinv, fwd);
  } else {
    if (ev_start)
      hipExtLaunchKernelGGL(k_lu_step_f64, dim3(n), dim3(256), step_lds<T>(), s, ev_start, ev_stop, 0, cp, cs, items,
                            refs, fops, K, Dinv, fwd);
    else
      hipLaunchKernelGGL(k_lu_step_f64, dim3(n), dim3(256), step_lds<T>(), s, cp, cs, items, refs, fops, K, Dinv,
                         fwd);
  }
}
void launch_lu_cell(hipStream_t s, const CellParams *cp, CellState *cs, const int2 *ranges, int ncell,
                    const StepItem *items, const BlockRef *refs, const FwdOp *fops, float *K, float *Dinv,
                    StepFwd<float> fwd, hipEvent_t ev_start, hipEvent_t ev_stop) {
  if (ncell <= 0) return;
  if (ev_start)
    hipExtLaunchKernelGGL(k_lu_cell_f32, dim3(ncell), dim3(256), 0, s, ev_start, ev_stop, 0, cp, cs, ranges, items,
                          refs, fops, K, Dinv, fwd);
  else
    hipLaunchKernelGGL(k_lu_cell_f32, dim3(ncell), dim3(256), 0, s, cp, cs, ranges, items, refs, fops, K, Dinv, fwd);
}

// ---------------------------------------------------------------------------
// Triangular sweeps, block LDU form (the lower factor has identity diagonal
// blocks, the upper one's diagonal inverses are in Dinv):
//   forward   y_b = r_b - sum_j L_bj y_j
//   backward  x_b = Dinv_b (y_b - sum_j U_bj x_j)
// One workgroup of 512 threads streams the blocks of its part of the plan in
// order (SweepOp): thread (row, part) = (tid / 8, tid % 8) owns eight columns
// of one row of each block, and SWEEP_RING blocks are in flight in registers
// ahead of the one being applied, across LDS-only barriers (a full
// __syncthreads also waits for outstanding global loads, which would
// serialise the stream).  What bounds a part is its stream (a compute unit
// sustains 60 to 110 GB/s) and two LDS barriers per block row, so a cell's
// leaves run in workgroups of their own: a forward launch over the leaves, a
// launch over the separators (forward and backward), a backward launch over
// the leaves.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
constexpr int SWEEP_THREADS = 512;
template <class T> struct SweepRing { static constexpr int v = 12; };
template <> struct SweepRing<double> { static constexpr int v = 6; };

// Column of a sweep thread's e-th entry (e = 0..7) of a 64-wide block row.
// FP32: columns 4q .. 4q+3 and 32+4q .. 32+4q+3 (two float4), so each load
// instruction of a wave takes whole 128-byte row segments; FP64: 2q, 2q+1 of
// each 16-column group (four double2, the same segments).
template <class T> __device__ __forceinline__ void row8_load(T (&v)[8], const T *row, int q) {
  if constexpr (sizeof(T) == 4) {
    const float4 a = *reinterpret_cast<const float4 *>(row + 4 * q);
    const float4 b = *reinterpret_cast<const float4 *>(row + 32 + 4 * q);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const double2 a = *reinterpret_cast<const double2 *>(row + 16 * g + 2 * q);
      v[2 * g] = a.x;
      v[2 * g + 1] = a.y;
    }
  }
}
// sum over the 8 lanes of each aligned group, in every lane.  FP32 by DPP
// (quad_perm 1,0,3,2 and 2,3,0,1, then row_half_mirror: lane i adds the other
// quad's sum).
template <class T> __device__ __forceinline__ T sum8(T v) {
  if constexpr (sizeof(T) == 4) {
    auto dpp = [](float x, auto ctrl) {
      return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xF, 0xF, false));
    };
    v += dpp(v, std::integral_constant<int, 0xB1>{});
    v += dpp(v, std::integral_constant<int, 0x4E>{});
    v += dpp(v, std::integral_constant<int, 0x141>{});
    return v;
  } else {
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    return v;
  }
}

// One part by the workgroup; y: its LDS vector, rowb: 64 entries of LDS.
template <class T>
__device__ __forceinline__ void sweep_part(const CellParams &p, const SweepPart &pt, const SweepOp *ops,
                                           const SweepLoc *locs, const int *accs, const T *K, const T *Dinv,
                                           const int *kinv, const SweepVec<T> &sv, int accumulate, T *y, T *rowb) {
  constexpr int RING = SweepRing<T>::v;
  const long long ld = p.npad;
  const int r = threadIdx.x >> 3, q = threadIdx.x & 7, nop = pt.nop;
  const T *A = K + p.k_off + (long long)r * ld;
  const T *D = Dinv + dinv_off(p, 0) + 4096 + r * 64;
  const int4 *op = reinterpret_cast<const int4 *>(ops + pt.op0);
  const SweepLoc *loc = locs + pt.loc0;
  T *slots = sv.slot + (long long)p.slot_off * NB;
  // The operations themselves: lane l of every wave holds operation l of the
  // current chunk and of the next, and the one needed is broadcast by lane
  // reads (a load per operation would put a memory round trip on each).
  // Every load of the loop is unconditional (past the end: block (0, 0)): a
  // load under a branch makes the compiler wait for all outstanding ones.
  constexpr int CHUNK = 5 * RING;
  const int lane = threadIdx.x & 63;
  auto op_load = [&](int o) {
    const int4 v = op[min(o + lane, nop > 0 ? nop - 1 : 0)];
    return o + lane < nop ? v : make_int4(0, 0, 0, 0);
  };
  int4 cur = op_load(0), nxt = op_load(CHUNK);
  T R[RING][8];
  auto fetch = [&](T(&v)[8], int l) {
    const bool n = l >= CHUNK;
    const int m = n ? l - CHUNK : l;
    const int x = __builtin_amdgcn_readlane(n ? nxt.x : cur.x, m), w = __builtin_amdgcn_readlane(n ? nxt.w : cur.w, m);
    const int bi = x & 0xFFFF, bj = x >> 16;
    row8_load<T>(v, w ? D + (long long)bi * 8192 : A + blk_off(bi, bj, ld), q);
  };
#pragma unroll
  for (int i = 0; i < RING; ++i) fetch(R[i], i);
  for (int i = threadIdx.x; i < pt.nloc * 64; i += SWEEP_THREADS) {
    const SweepLoc l = loc[i >> 6];
    const int row = p.sys_off + l.b * NB + (i & 63);
    T v;
    if (l.init == SL_RHS && !sv.from_y) {
      const int dof = kinv[row];
      v = dof >= 0 ? (T)sv.rhs[dof] : T(0);
      for (int a = 0; a < l.nacc; ++a) v -= slots[(long long)accs[l.acc0 + a] * NB + (i & 63)];
    } else {
      v = (l.init == SL_X ? sv.x : sv.y)[row];
    }
    y[i] = v;
  }
  lds_barrier();
  T part = T(0);
  for (int c0 = 0; c0 < nop; c0 += CHUNK) {
    for (int l0 = 0; l0 < CHUNK && c0 + l0 < nop; l0 += RING) {
#pragma unroll
      for (int i = 0; i < RING; ++i) {
        const int l = l0 + i;
        const int w1 = __builtin_amdgcn_readlane(cur.y, l), dst = __builtin_amdgcn_readlane(cur.z, l);
        const int vec = (int)(int16_t)(w1 & 0xFFFF), kind = c0 + l < nop ? w1 >> 16 : SW_SUM;
        T v[8];
        row8_load<T>(v, vec < 0 ? rowb : y + vec * NB, q);
#pragma unroll
        for (int e = 0; e < 8; ++e) part += R[i][e] * v[e];
        if (kind != SW_SUM) {
          part = sum8(part);
          if (kind == SW_FWD) {
            if (q == 0) y[dst * NB + r] -= part;
            lds_barrier();
          } else if (kind == SW_BSUM) {
            if (q == 0) rowb[r] = y[dst * NB + r] - part;
            lds_barrier();
          } else if (kind == SW_DIAG) {
            if (vec >= 0) lds_barrier();  // no later block: y_dst itself was multiplied, read before it is replaced
            if (q == 0) y[dst * NB + r] = part;
            lds_barrier();
          } else if (q == 0) {
            slots[(long long)dst * NB + r] = part;
          }
          part = T(0);
        }
        fetch(R[i], l + RING);
      }
    }
    cur = nxt;
    nxt = op_load(c0 + 2 * CHUNK);
  }
  lds_barrier();
  for (int i = threadIdx.x; i < pt.nloc * 64; i += SWEEP_THREADS) {
    const SweepLoc l = loc[i >> 6];
    const int row = p.sys_off + l.b * NB + (i & 63);
    if (l.out & SL_OUT_Y) sv.x[row] = y[i];
    if (l.out & SL_OUT_D) {
      const int dof = kinv[row];
      if (dof >= 0) sv.delta[dof] = accumulate ? sv.delta[dof] + (double)y[i] : (double)y[i];
    }
  }
}
template <class T>
__global__ __launch_bounds__(SWEEP_THREADS) void k_band_sweep(const CellParams *cp, const CellState *cs,
                                                              const SweepWG *wgs, const SweepOp *ops,
                                                              const SweepLoc *locs, const int *accs, const T *K,
                                                              const T *Dinv, const int *kinv, SweepVec<T> sv,
                                                              int accumulate) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ __attribute__((aligned(16))) T rowb[64];
  const SweepWG wg = wgs[blockIdx.x];
  if (cs[wg.cell].ir_done) return;
  sweep_part<T>(cp[wg.cell], wg.part, ops, locs, accs, K, Dinv, kinv, sv, accumulate, reinterpret_cast<T *>(smem),
                rowb);
}

// sum over a cell's boundary vertices of g . v
__device__ __forceinline__ double boundary_gdot(const CellParams &p, const BndView &bv, const double *v, double *red) {
  double a = 0.0;
  for (int b = p.bnd_off + threadIdx.x; b < p.bnd_off + p.n_bnd; b += SWEEP_THREADS) {
    if (bv.frame[b].x < 0) continue;
    const double2 g = bv.g[b], d = reinterpret_cast<const double2 *>(v)[bv.node[b]];
    a += g.x * d.x + g.y * d.y;
  }
  return block_sum<SWEEP_THREADS>(a, red);
}
// A cell with smw: its step inc - z t as direction nd (P0: the cell's
// directions), orthogonal (its K times) to the ones before it, and delta along
// it to the least residual; false: no direction.  A function of its own with
// its arguments in memory: inline it took the sweeps' registers (905-element
// cell, load step: 8 us).
__device__ __attribute__((noinline)) bool refine_direction(const RefineArgs *args, const CellParams *cp, double *P0, int nd,
                                                           double t, double *red) {
  const RefineArgs &ra = *args;
  const CellParams &p = *cp;
  const int n0 = p.node_off, n2 = 2 * p.n_nodes;
  double *P = P0 + 2LL * nd * n2, *Q = P + n2;
  for (int i = threadIdx.x; i < n2; i += SWEEP_THREADS) {
    const double d = ra.inc[2 * n0 + i];
    P[i] = t != 0.0 ? d - ra.z[2 * n0 + i] * t : d;
  }
  __syncthreads();
  const double gd = boundary_gdot(p, ra.bv, P - 2 * n0, red);
  for (int i = threadIdx.x; i < p.n_nodes; i += SWEEP_THREADS) {
    const double2 q = product_node(n0 + i, ra.el_tri, ra.adj_start, ra.adj, ra.Ke64, P - 2 * n0, p, ra.bv, gd);
    Q[2 * i] = q.x;
    Q[2 * i + 1] = q.y;
  }
  __syncthreads();
  auto dot = [&](const double *a, const double *b) {
    double v = 0.0;
    for (int i = threadIdx.x; i < n2; i += SWEEP_THREADS) v += a[i] * b[i];
    return block_sum<SWEEP_THREADS>(v, red);
  };
#pragma unroll 1
  for (int k = 0; k < 2 * nd; ++k) {  // twice: one pass leaves what cancellation made
    const double *Pk = P0 + 2LL * (k % nd) * n2, *Qk = Pk + n2;
    const double a = dot(Qk, Q);
    for (int i = threadIdx.x; i < n2; i += SWEEP_THREADS) {
      P[i] -= a * Pk[i];
      Q[i] -= a * Qk[i];
    }
  }
  const double qq = dot(Q, Q), s = 1.0 / sqrt(qq);
  if (!(qq > 0.0 && s > 0.0)) return false;  // nothing new, or not finite
  const double a = s * s * dot(Q, ra.r + 2 * n0);
  for (int i = threadIdx.x; i < n2; i += SWEEP_THREADS) {
    ra.delta[2 * n0 + i] += a * P[i];
    P[i] *= s;
    Q[i] *= s;
  }
  __syncthreads();
  return true;
}

// The whole refinement of one cell: sweep, FP64 residual, norm and control,
// again until lin_rtol is met.  Small cells: a sweep streams few blocks, so
// five launches per refinement sweep (also of the sweeps that have nothing
// left to do: 4.5 us each in a captured graph) cost more than the work.
// Cells with smw: the system in the band is B = K - k g g^T (the area term's
// rank one left out, g = dA/dx on the boundary), and K d = r is solved as
// d = y - z (g.y) / (1 + g.z) with y = B^-1 r, z = B^-1 k g (Sherman and
// Morrison 1950), the dots in FP64; the residual is the full K's.  The full
// matrix is dense (the boundary couples to itself): n^3 instead of n bw^2
// (905 elements, load step of two to three Newton steps: 1600 -> 610 us).
// z stays as the factors give it: refined against B it would no longer belong
// to the matrix that was factored (B with rounding and replaced pivots).
// B can be singular where K is not (the area off area_0 by a pressure that the
// cell's stiffness balances); then y and z are large, almost cancel, and the
// sweeps stall.  From the first sweep that leaves more than REFINE_POOR of the
// residual, or a last one (of max_refine) that leaves more than roundoff
// explains (1e-2, FP64 1e-4), the solve is mixed block
// elimination (Govaerts and Pryce 1990; its solve with the transpose taken as
// z / k, which the mostly symmetric B allows): a first guess of the rank one's
// part leaves the right-hand side before B^-1 is applied.  The updates then are
// search directions (generalized conjugate residuals, Eisenstat, Elman and
// Schultz 1983): of all their combinations the one of least residual, so that
// what is left wrong in a few directions costs a sweep each.  At most
// REFINE_MORE sweeps above max_refine; with B singular to rounding and K of
// condition 2e3 to 4e5 three to six in all to 1e-8, where sweeps by the rank
// one formula alone stood at 0.03 to 0.8 of the residual after four.
constexpr double REFINE_POOR = 1.0 / 16.0, REFINE_FLOOR = 1e-13;  // FLOOR: rounding of the FP64 residual
// SMW: a batch with cells with smw (without them the kernel holds neither path
// of theirs: 1.5 % of the 905-element FP64 step).
template <class T, bool SMW>
__global__ __launch_bounds__(SWEEP_THREADS) void k_band_refine(const CellParams *cp, CellState *cs,
                                                               const RefineWG *wgs, const SweepOp *ops,
                                                               const SweepLoc *locs, const int *accs, const T *K,
                                                               const T *Dinv, const int *kinv, SweepVec<T> sv,
                                                               RefineArgs ra) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ __attribute__((aligned(16))) T rowb[64];
  __shared__ double red[SWEEP_THREADS];
  __shared__ int done;
  T *y = reinterpret_cast<T *>(smem);
  const RefineWG wg = wgs[blockIdx.x];
  const int c = wg.cell;
  if (cs[c].ir_done) return;
  const CellParams &p = cp[c];
  const int n0 = p.node_off, n1 = n0 + p.n_nodes;
  auto gdot = [&](const double *v) { return boundary_gdot(p, ra.bv, v, red); };
  auto g_of = [&](int i) {
    const int b = ra.bv.bidx[i];
    return b >= 0 && ra.bv.frame[b].x >= 0 ? ra.bv.g[b] : make_double2(0.0, 0.0);
  };
  const bool smw = SMW && p.smw;
  if (smw) {  // the first sweep below: z = B^-1 k g
    for (int i = n0 + threadIdx.x; i < n1; i += SWEEP_THREADS) {
      const double2 g = g_of(i);
      ra.inc[2 * i] = p.k_area * g.x;
      ra.inc[2 * i + 1] = p.k_area * g.y;
    }
    __syncthreads();
  }
  double den = 1.0;
  bool rank1 = true;
  if (ra.it0 == 0 && !ra.fwd_done) {
    for (int i = 2 * n0 + threadIdx.x; i < 2 * n1; i += SWEEP_THREADS) ra.r[i] = -ra.G[i];
    __syncthreads();
  }
  auto residual = [&]() {  // r, and its squared norm
    const double gd = p.bterm & BT_AREA ? gdot(ra.delta) : 0.0;
    double rr = 0.0;
    for (int i = n0 + threadIdx.x; i < n1; i += SWEEP_THREADS) {
      const double2 ri = residual_node(i, ra.el_tri, ra.adj_start, ra.adj, ra.Ke64, ra.G, ra.delta, p, ra.bv, gd);
      ra.r[2 * i] = ri.x;
      ra.r[2 * i + 1] = ri.y;
      rr += ri.x * ri.x + ri.y * ri.y;
    }
    return block_sum<SWEEP_THREADS>(rr, red);
  };
  auto step = [&](int i, double t) { return t != 0.0 ? ra.inc[i] - ra.z[i] * t : ra.inc[i]; };
  int nd = -1;  // cells with smw: directions so far (refine_direction); -1: plain refinement
  const double bnorm = cs[c].bnorm, slow = sizeof(T) == 4 ? 1e-2 : 1e-4;
  double last = bnorm, y1 = 0.0;  // y1: the first guess of g . d
  int most = ra.max_refine;
  for (int it = smw ? ra.it0 - 1 : ra.it0; it < most; ++it) {
    const bool zsweep = smw && it < ra.it0;
    SweepVec<T> v = sv;
    v.rhs = zsweep ? ra.inc : ra.r;
    v.from_y = it == 0 && ra.fwd_done ? 1 : 0;
    v.delta = zsweep ? ra.z : smw ? ra.inc : ra.delta;
    if (smw && nd >= 0) {
      double s = 0.0;
      for (int i = 2 * n0 + threadIdx.x; i < 2 * n1; i += SWEEP_THREADS) s += ra.z[i] * ra.r[i];
      s = rank1 ? block_sum<SWEEP_THREADS>(s, red) / den : 0.0;
      y1 = s / p.k_area;
      for (int i = n0 + threadIdx.x; i < n1; i += SWEEP_THREADS) {
        const double2 g = g_of(i);
        ra.inc[2 * i] = ra.r[2 * i] - g.x * s;
        ra.inc[2 * i + 1] = ra.r[2 * i + 1] - g.y * s;
      }
      __syncthreads();
      v.rhs = ra.inc;
    }
    sweep_part<T>(p, v.from_y ? wg.bwd : wg.whole, ops, locs, accs, K, Dinv, kinv, v, smw ? 0 : it > 0, y, rowb);
    __syncthreads();
    if (zsweep) {
      den = 1.0 + gdot(ra.z);
      rank1 = fabs(den) > 0.0 && fabs(den) < 1e300;
      continue;
    }
    const double t = smw && rank1 ? (gdot(ra.inc) - y1) / den : 0.0;
    bool stop = false, undone = false;
    if (smw && nd >= 0) {
      stop = !refine_direction(ra.mem, &p, ra.dirs + wg.dirs, nd, t, red);
      if (!stop) nd = nd + 1 < REFINE_DIRS ? nd + 1 : 0;
      if (stop && rank1) rank1 = stop = false;  // without the rank one: B alone, one direction more
    } else if (smw) {
      for (int i = 2 * n0 + threadIdx.x; i < 2 * n1; i += SWEEP_THREADS) {
        const double d = step(i, t);
        ra.delta[i] = it > 0 ? ra.delta[i] + d : d;
      }
      __syncthreads();
    }
    double nrm;
#pragma unroll 1
    for (;;) {
      nrm = sqrt(residual());
      if (!smw || nd >= 0 || undone) break;
      const bool poor = !(nrm <= ra.lin_rtol * bnorm) && !(nrm <= REFINE_FLOOR * bnorm) &&
                        (!(nrm <= REFINE_POOR * last) || (it + 1 == ra.max_refine && !(nrm <= slow * last)));
      if (poor) most = ra.max_refine + REFINE_MORE;
      if (poor && !(nrm <= last)) {  // worse than before the sweep: without it
        for (int i = 2 * n0 + threadIdx.x; i < 2 * n1; i += SWEEP_THREADS) {
          const double b = it > 0 ? ra.delta[i] - step(i, t) : 0.0;
          ra.delta[i] = fabs(b) < 1e300 ? b : 0.0;
        }
        __syncthreads();
        undone = true;
        continue;
      }
      last = nrm;
      if (poor) nd = 0;
      break;
    }
    if (undone) nd = 0;
    if (threadIdx.x == 0) {
      CellState &s = cs[c];
      norm_finish(s, 1, nrm, ra.lin_rtol);
      done = s.ir_done;
    }
    __syncthreads();
    if (done || stop) return;
  }
}
size_t refine_max_dynamic(size_t max_lds) { return max_lds > 8192 ? max_lds - 8192 : 0; }
template <class T>
void launch_band_refine(hipStream_t s, const CellParams *cp, CellState *cs, const RefineWG *wgs, int nwg, int max_loc,
                        const SweepOp *ops, const SweepLoc *locs, const int *accs, const T *K, const T *Dinv,
                        const int *kinv, const SweepVec<T> &sv, const RefineArgs &ra) {
  if (nwg <= 0) return;
  const auto k = ra.dirs ? &k_band_refine<T, true> : &k_band_refine<T, false>;
  hipLaunchKernelGGL(k, dim3(nwg), dim3(SWEEP_THREADS), (size_t)max_loc * NB * sizeof(T), s, cp, cs, wgs, ops, locs,
                     accs, K, Dinv, kinv, sv, ra);
}
template <class T>
void launch_band_sweep(hipStream_t s, const CellParams *cp, const CellState *cs, const SweepWG *wgs, int nwg,
                       int max_loc, const SweepOp *ops, const SweepLoc *locs, const int *accs, const T *K,
                       const T *Dinv, const int *kinv, const SweepVec<T> &sv, int accumulate) {
  if (nwg <= 0) return;
  hipLaunchKernelGGL(k_band_sweep<T>, dim3(nwg), dim3(SWEEP_THREADS), (size_t)max_loc * NB * sizeof(T), s, cp, cs, wgs,
                     ops, locs, accs, K, Dinv, kinv, sv, accumulate);
}

hipError_t band_prepare_attributes(size_t max_lds) {
  const int dyn = (int)lu_solve_max_dynamic(max_lds);
  const int ref = (int)refine_max_dynamic(max_lds);
  const std::pair<const void *, int> fns[] = {{reinterpret_cast<const void *>(&k_band_refine<float, false>), ref},
                                              {reinterpret_cast<const void *>(&k_band_refine<float, true>), ref},
                                              {reinterpret_cast<const void *>(&k_band_refine<double, false>), ref},
                                              {reinterpret_cast<const void *>(&k_band_refine<double, true>), ref},
                                              {reinterpret_cast<const void *>(&k_band_sweep<float>), dyn},
                                              {reinterpret_cast<const void *>(&k_band_sweep<double>), dyn},
                                              {reinterpret_cast<const void *>(&k_lu_step_f64), step_lds<double>()}};
  for (const auto &f : fns) {
    hipError_t e = hipFuncSetAttribute(f.first, hipFuncAttributeMaxDynamicSharedMemorySize, f.second);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

#define WCFE_INST(T)                                                                                                \
  template void launch_lu_step<T>(hipStream_t, const CellParams *, CellState *, const StepItem *, int,               \
                                  const BlockRef *, const FwdOp *, T *, T *, StepFwd<T>, hipEvent_t, hipEvent_t);    \
  template void launch_band_sweep<T>(hipStream_t, const CellParams *, const CellState *, const SweepWG *, int, int,  \
                                     const SweepOp *, const SweepLoc *, const int *, const T *, const T *,          \
                                     const int *, const SweepVec<T> &, int);                                        \
  template void launch_band_refine<T>(hipStream_t, const CellParams *, CellState *, const RefineWG *, int, int,      \
                                      const SweepOp *, const SweepLoc *, const int *, const T *, const T *,         \
                                      const int *, const SweepVec<T> &, const RefineArgs &);
WCFE_INST(float)
WCFE_INST(double)

}  // namespace wcfe
