// Checks band plans (wholecellfe_amd/csrc/band_plan.hpp) on the CPU: every
// launch's items are run on the values from before the launch (so an item
// that reads what another writes is found), on random band matrices with
// 2 x 2 blocks, and the sweeps' solutions are put back into the matrix.
#include "../wholecellfe_amd/csrc/band_plan.hpp"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>

using namespace wcfe;
typedef std::vector<double> Vec;
constexpr int B = 2;

static void die(const char *what, int n, int bw, int sym, int cuts) {
  std::printf("%s: n %d bw %d sym %d cuts %d\n", what, n, bw, sym, cuts);
  std::exit(1);
}

static void check(int n, int bw, int sym, int cuts, std::mt19937 &rng) {
  std::normal_distribution<double> nd;
  const BandPlan P = make_band_plan(n, bw, sym, cuts);
  if ((int)P.lev.size() != band_steps(n, bw, cuts)) die("band_steps differs", n, bw, sym, cuts);
  const int N = n * B;
  Vec A0(N * N, 0.0), A(N * N, NAN), rhs(N), y(N, NAN), slot(P.nslot * B, NAN);
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < N; ++j)
      if (std::abs(i / B - j / B) <= bw) A0[i * N + j] = sym && j < i ? A0[j * N + i] : nd(rng);
  for (int i = 0; i < N; ++i) A0[i * N + i] += 4.0 * (bw + 1) * B;
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < N; ++j)
      if (std::abs(i / B - j / B) <= bw && (!sym || P.rank[i / B] >= P.rank[j / B])) A[i * N + j] = A0[i * N + j];
  for (double &v : rhs) v = nd(rng);
  std::vector<Vec> D(n);
  auto get = [&](const Vec &M, int i, int j) {
    Vec m(B * B);
    for (int r = 0; r < B; ++r)
      for (int c = 0; c < B; ++c) m[r * B + c] = M[(i * B + r) * N + j * B + c];
    return m;
  };
  auto mul = [](const Vec &x, const Vec &z) {
    Vec o(B * B, 0.0);
    for (int r = 0; r < B; ++r)
      for (int c = 0; c < B; ++c)
        for (int k = 0; k < B; ++k) o[r * B + c] += x[r * B + k] * z[k * B + c];
    return o;
  };
  for (const BandPlan::Level &L : P.lev) {
    const Vec A1 = A, y1 = y, slot1 = slot;
    std::set<std::pair<int, int>> wrote, read;
    std::set<int> wy, ry, ws, rs;
    auto rd = [&](int i, int j) {
      read.insert({i, j});
      return get(A1, i, j);
    };
    auto wr = [&](int i, int j, const Vec &m) {
      if (!wrote.insert({i, j}).second) die("two items write one block", n, bw, sym, cuts);
      for (int r = 0; r < B; ++r)
        for (int c = 0; c < B; ++c) A[(i * B + r) * N + j * B + c] = m[r * B + c];
    };
    auto update = [&](Vec &c, int i, int p, int j) {
      const Vec u = mul(rd(i, p), rd(p, j));
      for (int k = 0; k < B * B; ++k) c[k] -= u[k];
    };
    for (const BandPlan::Pivot &v : L.piv) {
      Vec d = rd(v.s, v.s);
      if (v.p >= 0) update(d, v.s, v.p, v.s);
      const double det = d[0] * d[3] - d[1] * d[2];
      D[v.s] = Vec{d[3] / det, -d[1] / det, -d[2] / det, d[0] / det};
      for (int q = 0; q < v.nref; ++q) {
        const BlockRef &r = P.refs[v.ref0 + q];
        Vec c = r.first ? Vec(B * B, 0.0) : get(A1, r.bi, r.bj);
        if (r.p0 >= 0) update(c, r.bi, r.p0, r.bj);
        if (sym) wr(v.s, r.bi, Vec{c[0], c[2], c[1], c[3]});
        wr(r.bi, v.s, mul(c, D[v.s]));
      }
    }
    for (const BandPlan::Group &g : L.grp) {
      for (int q = 0; q < g.nref; ++q) {
        const BlockRef &r = P.refs[g.ref0 + q];
        Vec c = r.first ? Vec(B * B, 0.0) : get(A1, r.bi, r.bj);
        for (int p : {(int)r.p0, (int)r.p1})
          if (p >= 0) update(c, r.bi, p, r.bj);
        wr(r.bi, r.bj, c);
      }
      double sum[B] = {0, 0};
      for (int q = 0; q < g.nfop; ++q) {
        const FwdOp &o = P.fops[g.fop0 + q];
        auto dot = [&](double *s) {
          const Vec l = rd(o.i, o.p);
          ry.insert(o.p);
          for (int r = 0; r < B; ++r)
            for (int c = 0; c < B; ++c) s[r] += l[r * B + c] * y1[o.p * B + c];
        };
        if (o.kind == FW_TERM) {
          dot(sum);
        } else if (o.kind == FW_SUB) {
          rs.insert(o.slot);
          for (int r = 0; r < B; ++r) sum[r] += slot1[o.slot * B + r];
        } else if (o.kind == FW_END) {
          wy.insert(o.i);
          for (int r = 0; r < B; ++r) {
            y[o.i * B + r] = rhs[o.i * B + r] - sum[r];
            sum[r] = 0.0;
          }
        } else {
          double s[B] = {0, 0};
          dot(s);
          if (!ws.insert(o.slot).second) die("two operations write one slot", n, bw, sym, cuts);
          for (int r = 0; r < B; ++r) slot[o.slot * B + r] = (o.kind == FW_ACC0 ? 0.0 : slot1[o.slot * B + r]) + s[r];
        }
      }
    }
    for (auto &x : read)
      if (wrote.count(x)) die("an item reads a block that another writes", n, bw, sym, cuts);
    for (int v : ry)
      if (wy.count(v)) die("an operation reads a row that another writes", n, bw, sym, cuts);
    for (int v : rs)
      if (ws.count(v)) die("an operation reads a slot that another writes", n, bw, sym, cuts);
  }
  auto sweep = [&](const SweepPart &S, const Vec &yin, Vec &x, Vec &sl, Vec &out, bool from_y) {
    Vec v(S.nloc * B);
    for (int l = 0; l < S.nloc; ++l) {
      const SweepLoc &q = P.locs[S.loc0 + l];
      for (int r = 0; r < B; ++r) {
        double t = q.init == SL_X ? x[q.b * B + r] : (q.init == SL_Y || from_y) ? yin[q.b * B + r] : rhs[q.b * B + r];
        if (q.init == SL_RHS && !from_y)
          for (int a = 0; a < q.nacc; ++a) t -= sl[P.accs[q.acc0 + a] * B + r];
        v[l * B + r] = t;
      }
    }
    double sum[B] = {0, 0}, row[B] = {NAN, NAN};
    for (int o = 0; o < S.nop; ++o) {
      const SweepOp &p = P.ops[S.op0 + o];
      const Vec m = p.inv ? D[p.bi] : get(A, p.bi, p.bj);
      const double *w = p.vec < 0 ? row : &v[p.vec * B];
      for (int r = 0; r < B; ++r)
        for (int c = 0; c < B; ++c) sum[r] += m[r * B + c] * w[c];
      if (p.kind == SW_SUM) continue;
      for (int r = 0; r < B; ++r) {
        if (p.kind == SW_FWD) v[p.dst * B + r] -= sum[r];
        if (p.kind == SW_BSUM) row[r] = v[p.dst * B + r] - sum[r];
        if (p.kind == SW_DIAG) v[p.dst * B + r] = sum[r];
        if (p.kind == SW_ACC) sl[p.dst * B + r] = sum[r];
        sum[r] = 0.0;
      }
    }
    for (int l = 0; l < S.nloc; ++l) {
      const SweepLoc &q = P.locs[S.loc0 + l];
      for (int r = 0; r < B; ++r) {
        if (q.out & SL_OUT_Y) x[q.b * B + r] = v[l * B + r];
        if (q.out & SL_OUT_D) out[q.b * B + r] = v[l * B + r];
      }
    }
  };
  auto solved = [&](const Vec &x, const char *what) {
    for (int i = 0; i < N; ++i) {
      double s = rhs[i];
      for (int j = 0; j < N; ++j) s -= A0[i * N + j] * x[j];
      if (!(std::fabs(s) < 1e-9)) die(what, n, bw, sym, cuts);
    }
  };
  Vec x(N, NAN), d(N, NAN), sl(P.nslot * B, NAN);
  if (P.top.nloc) sweep(P.top_bwd, y, x, sl, d, true);
  for (const SweepPart &S : P.bwd) sweep(S, y, x, sl, d, true);
  solved(d, "first solve");
  x.assign(N, NAN);
  d.assign(N, NAN);
  sl.assign(P.nslot * B, NAN);
  for (const SweepPart &S : P.fwd) sweep(S, x, x, sl, d, false);
  if (P.top.nloc) sweep(P.top, x, x, sl, d, false);
  for (const SweepPart &S : P.bwd) sweep(S, x, x, sl, d, false);
  solved(d, "refinement solve");
  if (P.root.nloc) {  // separator by separator
    x.assign(N, NAN);
    d.assign(N, NAN);
    sweep(P.root_bwd, y, x, sl, d, true);
    for (const auto &level : P.sep_bwd)
      for (const SweepPart &S : level) sweep(S, y, x, sl, d, true);
    for (const SweepPart &S : P.bwd) sweep(S, y, x, sl, d, true);
    solved(d, "first solve by separators");
    x.assign(N, NAN);
    d.assign(N, NAN);
    sl.assign(P.nslot * B, NAN);
    for (const SweepPart &S : P.fwd) sweep(S, x, x, sl, d, false);
    for (size_t q = P.sep_fwd.size(); q-- > 0;)
      for (const SweepPart &S : P.sep_fwd[q]) sweep(S, x, x, sl, d, false);
    sweep(P.root, x, x, sl, d, false);
    for (const auto &level : P.sep_bwd)
      for (const SweepPart &S : level) sweep(S, x, x, sl, d, false);
    for (const SweepPart &S : P.bwd) sweep(S, x, x, sl, d, false);
    solved(d, "refinement solve by separators");
  }
  if (P.whole.nloc) {
    d.assign(N, NAN);
    sweep(P.whole_bwd, y, x, sl, d, true);
    solved(d, "first solve in one part");
    d.assign(N, NAN);
    sweep(P.whole, x, x, sl, d, false);
    solved(d, "one-part solve");
  }
}

int main() {
  std::mt19937 rng(1);
  for (int bw = 0; bw <= 8; ++bw)
    for (int n : {1, 2, 3, 4, 5, 6, 7, 9, 12, 15, 16, 21, 30, 41, 64, 82})
      for (int sym = 0; sym < 2; ++sym)
        for (int cuts = 0; cuts <= 5; ++cuts)
          if (bw < n) check(n, bw, sym, cuts, rng);
  std::printf("ok\n");
  return 0;
}
