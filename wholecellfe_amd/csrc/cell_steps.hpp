// Per-node and per-cell pieces of the Newton step, shared by the batch-wide
// kernels (k_assemble.hip) and the one-workgroup-per-cell ones (k_band.hip,
// k_boundary.hip).
#pragma once
#include "wcfe_internal.hpp"

namespace wcfe {

// which: 0 residual after assembly (sets gnorm, bnorm and g0 at the first
// iterate), 1 refinement residual (rnorm, and the refinement control for
// lin_rtol >= 0), 2 residual after the update (gnorm)
__device__ __forceinline__ void norm_finish(CellState &s, int which, double nrm, double lin_rtol) {
  if (which == 0) {
    s.gnorm = nrm;
    s.bnorm = nrm;
    if (s.newton_it == 0) s.g0 = nrm;
    s.ir_done = 0;  // a new linear solve
    s.ir_iters = 0;
    s.lin_relres = 0.0;
  } else if (which == 1) {
    s.rnorm = nrm;
    if (lin_rtol >= 0.0 && !s.ir_done) {  // refinement control of this cell
      s.ir_iters += 1;
      s.lin_relres = s.bnorm > 0.0 ? s.rnorm / s.bnorm : 0.0;
      if (s.rnorm <= lin_rtol * s.bnorm) s.ir_done = 1;
    }
  } else {
    s.gnorm = nrm;
  }
}

// Static-pivot threshold of the factorization: 64 eps times the largest
// diagonal entry m.
__device__ __forceinline__ void tau_finish(CellState &s, double m, double eps) {
  s.tau = 64.0 * eps * (m > 0.0 ? m : 1.0);
  s.n_static = 0;
  s.zero_pivot = 0;
}

// The Newton convergence test after the update's residual norm.
__device__ __forceinline__ void newton_finish(CellState &s, double rtol, double atol) {
  s.newton_it += 1;
  s.converged = (s.gnorm <= rtol * s.g0 || s.gnorm <= atol) ? 1 : 0;
  if (!s.ir_done) s.lin_failed = 1;
}

// K d of one node, from the stored FP64 element matrices over its elements in
// element order, and the node terms (drag diagonal, the boundary vertex's
// 2 x 6 block, the area term's rank-one part k g_i (sum_m g_m . d_m), gd the
// sum).
__device__ __forceinline__ double2 product_node(int i, const int *el_tri, const int *adj_start, const int *adj,
                                                const double *Ke64, const double *delta, const CellParams &p,
                                                const BndView &bv, double gd) {
  const double2 *d2 = reinterpret_cast<const double2 *>(delta);
  double y0 = 0.0, y1 = 0.0;
  for (int k = adj_start[i]; k < adj_start[i + 1]; ++k) {
    const int pk = adj[k];
    const int e = pk >> 2, a = pk & 3;
    const double *Ke = Ke64 + 36 * (long long)e + 12 * a;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const double2 d = d2[el_tri[3 * e + b]];
      y0 += Ke[2 * b] * d.x + Ke[2 * b + 1] * d.y;
      y1 += Ke[6 + 2 * b] * d.x + Ke[6 + 2 * b + 1] * d.y;
    }
  }
  if (bv.bidx && p.bterm) {
    const double2 di = d2[i];
    if (p.bterm & BT_DRAG) {
      const double cd = p.drag / bv.dt;
      y0 += cd * di.x;
      y1 += cd * di.y;
    }
    const int b = bv.bidx[i];
    if (b >= 0 && (p.bterm & (BT_BEND | BT_AREA))) {
      const int2 fr = bv.frame[b];
      if (fr.x >= 0) {
        const double *J = bv.J + 12LL * b;
        const double2 d1 = d2[fr.x], dd2 = d2[fr.y];
        y0 += J[0] * di.x + J[1] * di.y + J[2] * d1.x + J[3] * d1.y + J[4] * dd2.x + J[5] * dd2.y;
        y1 += J[6] * di.x + J[7] * di.y + J[8] * d1.x + J[9] * d1.y + J[10] * dd2.x + J[11] * dd2.y;
        if (p.bterm & BT_AREA) {
          const double2 g = bv.g[b];
          y0 += p.k_area * g.x * gd;
          y1 += p.k_area * g.y * gd;
        }
      }
    }
  }
  return make_double2(y0, y1);
}
// r = -G - K d of one node
__device__ __forceinline__ double2 residual_node(int i, const int *el_tri, const int *adj_start, const int *adj,
                                                 const double *Ke64, const double *G, const double *delta,
                                                 const CellParams &p, const BndView &bv, double gd) {
  const double2 y = product_node(i, el_tri, adj_start, adj, Ke64, delta, p, bv, gd);
  return make_double2(-G[2 * i] - y.x, -G[2 * i + 1] - y.y);
}

// Sum over a workgroup of NT threads (a power of two), in every thread: a
// fixed tree.  red: NT doubles of LDS.
template <int NT> __device__ __forceinline__ double block_sum(double v, double *red) {
  __syncthreads();
  red[threadIdx.x] = v;
  __syncthreads();
#pragma unroll
  for (int w = NT / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  return red[0];
}

// Strain increment and lumped mass of one node of a UL cell, over its elements
// in element order.
__device__ __forceinline__ void node_strain(const View &v, int i, const int *adj_start, const int *adj, double *Rea,
                                            double *MM) {
  double re[3] = {0.0, 0.0, 0.0}, m = 0.0;
  for (int k = adj_start[i]; k < adj_start[i + 1]; ++k) {
    const int e = adj[k] >> 2, a = adj[k] & 3;
    double rea[9], mm[3];
    element_strain(v, e, rea, mm);
#pragma unroll
    for (int q = 0; q < 3; ++q) re[q] += a == 0 ? rea[q] : a == 1 ? rea[3 + q] : rea[6 + q];
    m += a == 0 ? mm[0] : a == 1 ? mm[1] : mm[2];
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) Rea[3 * i + q] = re[q];
  MM[i] = m;
}

// UL:607-612 strain update; UL:2046-2171 mean-field bond kinetics with a rigid
// substrate (subs_u = 0): fa_u += x - X, catch-slip k_off, forward Euler c_C,
// dissipative rescale; the new reference configuration is the converged x.
__device__ __forceinline__ void commit_node(const View &v, const CellParams &p, int i, double2 *X, const double2 *x,
                                            double *ea, double *cC, double2 *fau, const double *Rea, const double *MM,
                                            double dt) {
  if (p.law == LAW_UL) {
    const double m = MM[i];
    for (int q = 0; q < 3; ++q) ea[3 * i + q] += Rea[3 * i + q] / m;
  }
  const double2 xi = x[i], Xi = X[i];
  if (p.node_springs) {
    double2 u = fau[i];
    u.x = u.x + (xi.x - Xi.x);
    u.y = u.y + (xi.y - Xi.y);
    if (p.kinetics == KIN_MEANFIELD) {
#pragma clang fp contract(off)
      double force;
      if (p.spring_law == SPRING_LINEAR) {
        force = p.k_lin * sqrt(u.x * u.x + u.y * u.y);  // 2D norm, UL1:2077
      } else {
        double f[2], J[4];
        spring_force(v, p, u.x, u.y, f, J);
        force = sqrt(f[0] * f[0] + f[1] * f[1]);  // UL:2137
      }
      const double k_on = 1.0, ka = 0.004, kb = 10.0, Fa = 15.0, Fb = 15.0;  // UL:2139-2143
      const double k_off = ka * shared_exp(force / Fa) + kb * shared_exp(-force / Fb);
      const double cold = cC[i];
      double cnew = cold + dt * k_on * (1.0 - cold) - dt * k_off * cold;
      if (cnew < 0.0) cnew = 0.0;
      cC[i] = cnew;
      const double keep = cold - dt * k_off * cold;
      if (keep > 0.0 && cnew > 0.0) {
        u.x = u.x * keep / cnew;
        u.y = u.y * keep / cnew;
      } else {
        u.x = 0.0 * u.x;
        u.y = 0.0 * u.y;
      }
    }
    fau[i] = u;
  }
  if (p.law == LAW_UL) X[i] = xi;
}

// Bell kinetics per barycentric spring after a converged load step:
// bound -> unbound with p = 1 - exp(-k_off0 e^{|F(D)|/f_b} dt), D = |u|,
// unbound -> bound
// with p = 1 - exp(-k_on dt), re-anchored at the current attachment point.
// Uniform u = (w + 0.5) 2^-32, w = Philox(ctr = (replica, spring, step, 0)).
__device__ __forceinline__ void commit_spring(const View &v, const CellParams &p, int c, unsigned step, int s,
                                              const int *sp_elem, const int *sp_local, double *state, double *anchor,
                                              const BellArgs &bell) {
  const int e = sp_elem[s];
  const double *bb = v.sp_bary + 3 * s;
  // attachment point (b0 x0 + b1 x1) + b2 x2, rounded term by term without
  // contraction so a re-anchored bond lands on the same bits as a plain FP64
  // evaluation of the same expression
  const double2 x0 = v.x[v.el_tri[3 * e]], x1 = v.x[v.el_tri[3 * e + 1]], x2 = v.x[v.el_tri[3 * e + 2]];
  double px, py;
  {
#pragma clang fp contract(off)
    px = bb[0] * x0.x + bb[1] * x1.x + bb[2] * x2.x;
    py = bb[0] * x0.y + bb[1] * x1.y + bb[2] * x2.y;
  }
  unsigned ctr[4] = {(unsigned)bell.replica[c], (unsigned)sp_local[s], step, 0u};
  philox4x32_10(ctr, bell.key_lo, bell.key_hi);
  const double u = ((double)ctr[0] + 0.5) * (1.0 / 4294967296.0);
  // the force and both probabilities rounded as written, with the shared exp
  if (state[s] != 0.0) {
    double ux, uy;
    {
#pragma clang fp contract(off)
      ux = px - anchor[2 * s];
      uy = py - anchor[2 * s + 1];
    }
    const double F = spring_magnitude(v, p, ux, uy);
    const double koff = bell.k_off0 * shared_exp(F / bell.f_b);
    const double prob = 1.0 - shared_exp(-koff * bell.dt);
    if (u < prob) {
      state[s] = 0.0;
      atomicAdd(bell.transitions, 1);
    }
  } else {
    const double prob = 1.0 - shared_exp(-bell.k_on * bell.dt);
    if (u < prob) {
      state[s] = 1.0;
      anchor[2 * s] = px;
      anchor[2 * s + 1] = py;
      atomicAdd(bell.transitions, 1);
    }
  }
}

}  // namespace wcfe
