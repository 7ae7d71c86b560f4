// Host-side plan of the band factorization of one cell: which 64 x 64 blocks
// are eliminated in which launch, the blocks each launch updates, and the
// triangular sweeps over the factors.  Plain C++ (no HIP types), so that a
// plan can be checked on the CPU.
//
// A band matrix of n block rows (block bandwidth bw) is cut by separators of
// bw consecutive blocks into a binary tree: removing a separator leaves two
// independent bands.  The leaves are eliminated at the same time, block by
// block; a separator's blocks follow when both sides are done.  With one leaf
// this is the plain top-down band LU (n dependent block steps), with two it is
// eliminated from both ends, with 2^d leaves about n / 2^d + d bw steps.  An
// inner leaf's pivots also update the separator above it (the fill of the
// cut): about three times the products per step, on compute units that a
// single chain leaves idle.
//
// Everything below is read off the symbolic elimination in that order: the
// structure of a pivot's column is every later block that the band or an
// earlier pivot's update couples to it, so the plan holds for any order in
// which the pivots of one level are independent.
#pragma once
#include <algorithm>
#include <cstdint>
#include <map>
#include <stdexcept>
#include <utility>
#include <vector>

namespace wcfe {

// A block update: A(bi, bj) -= L(bi, p) U(p, bj) for p0 and p1 (-1: none);
// first: the block is fill that nothing has written yet (taken as zero).
struct BlockRef {
  int16_t bi, bj, p0, p1;
  int32_t first, pad;
};
// Forward substitution of the first solve, run beside the block steps.
enum : int { FW_TERM = 0, FW_SUB = 1, FW_END = 2, FW_ACC0 = 3, FW_ACC = 4 };
struct FwdOp {
  int16_t kind, i, p, pad;  // TERM: sum += L(i, p) y_p; SUB: sum += slot; END: y_i = b_i - sum
  int32_t slot, pad2;       // ACC0 / ACC: slot (+)= L(i, p) y_p
};
// One workgroup's work in a block step launch.
enum : int { STEP_INV = 1, STEP_STORE = 2 };
struct StepItem {
  // INV: invert block s (after pivot p's update, -1: none), STORE the inverse,
  // then L(bi, s) = A(bi, s) A(s, s)^-1 for the refs; else update the refs'
  // blocks; then the forward operations
  int32_t cell, kind, s, p, ref0, nref, fop0, nfop;
};
// One 64 x 64 block of a triangular sweep, in the order a workgroup streams
// them: sum += M v with M = A(bi, bj) or the inverse of diagonal block bi, v a
// 64-entry block of the workgroup's LDS vector.  kind: what ends a row.
enum : int { SW_SUM = 0, SW_FWD = 1, SW_BSUM = 2, SW_DIAG = 3, SW_ACC = 4 };
struct SweepOp {
  int16_t bi, bj, vec, kind;  // vec < 0: the row buffer that BSUM wrote
  int32_t dst, inv;           // FWD: v_dst -= sum; BSUM: row = v_dst - sum; DIAG: v_dst = sum; ACC: slot dst = sum
};
// A block of a sweep workgroup's LDS vector.
enum : int { SL_RHS = 0, SL_Y = 1, SL_X = 2 };
enum : int { SL_OUT_Y = 1, SL_OUT_D = 2 };
struct SweepLoc {
  int32_t b, init, out, acc0, nacc, pad[3];  // RHS: minus the listed slots
};
struct SweepPart {
  int32_t op0 = 0, nop = 0, loc0 = 0, nloc = 0;
};

struct BandPlan {
  struct Pivot {
    int s, p, ref0, nref, node;
  };
  struct Group {  // blocks and forward operations of one node in one level
    int ref0, nref, fop0, nfop;
  };
  struct Count {  // pivots, or groups, with nref blocks (groups: with or without forward operations)
    int nref, fwd, n;
  };
  static void count(std::vector<Count> &c, int nref, int fwd, int n) {
    for (Count &q : c)
      if (q.nref == nref && q.fwd == fwd) {
        q.n += n;
        return;
      }
    c.push_back(Count{nref, fwd, n});
  }
  struct Level {
    std::vector<Pivot> piv;
    std::vector<Group> grp;
    std::vector<Count> pivs, grps;  // the same, counted
    long long products = 0;
  };
  int n = 0, bw = 0, leaves = 1, nslot = 0;
  bool sym = false;
  std::vector<int> rank;  // per block: its place in the elimination order
  std::vector<Level> lev;
  std::vector<BlockRef> refs;
  std::vector<FwdOp> fops;
  // sweeps: per leaf its forward and backward part; the separators' part
  // (forward and backward, or backward only), or (three and more separators)
  // one part per separator, by the number of cuts above it, the first cut's
  // forward and backward in one; the whole sweep by one workgroup
  std::vector<SweepPart> fwd, bwd;
  SweepPart top, top_bwd, root, root_bwd, whole, whole_bwd;
  std::vector<std::vector<SweepPart>> sep_fwd, sep_bwd;  // [0] empty
  std::vector<SweepOp> ops;
  std::vector<SweepLoc> locs;
  std::vector<int> accs;
};

namespace band_detail {
struct Node {
  int lo, hi, desc, leaf, start, lvl;  // lvl: cuts above it
};
// last level of a band of len blocks cut `depth` times, and the left part's length
inline int last_level(int len, int depth, int bw, std::map<std::pair<int, int>, std::pair<int, int>> &memo) {
  if (depth == 0 || len < bw + 2) return len - 1;
  auto it = memo.find({len, depth});
  if (it != memo.end()) return it->second.first;
  const int inner = len - bw;
  int best = 1 << 30, at = 0;
  for (int a = (inner + 1) / 2; a <= std::min(inner - 1, (inner + 1) / 2 + 2); ++a) {
    const int l = last_level(a, depth - 1, bw, memo), r = last_level(inner - a, depth - 1, bw, memo);
    // two sides that end together would leave two updates pending on the
    // separator's first block: it starts one level later then
    const int e = std::max(l, r) + (l == r ? 2 : 1) + bw - 1;
    if (e < best) { best = e; at = a; }
  }
  if (best >= len - 1) { best = len - 1; at = 0; }  // no shorter than one chain
  memo[{len, depth}] = {best, at};
  return best;
}
inline int cut(std::vector<Node> &nodes, int lo, int hi, int depth, int bw, bool hasl, bool hasr,
               std::map<std::pair<int, int>, std::pair<int, int>> &memo, int lvl = 0) {
  const int len = hi - lo;
  last_level(len, depth, bw, memo);
  auto it = memo.find({len, depth});
  if (depth == 0 || it == memo.end() || it->second.second == 0) {
    nodes.push_back(Node{lo, hi, hasl && !hasr ? 1 : 0, 1, 0, lvl});
    return len - 1;
  }
  const int a = it->second.second, m = lo + a;
  const int l = cut(nodes, lo, m, depth - 1, bw, hasl, true, memo, lvl + 1);
  const int r = cut(nodes, m + bw, hi, depth - 1, bw, true, hasr, memo, lvl + 1);
  const int start = std::max(l, r) + (l == r ? 2 : 1);
  nodes.push_back(Node{m, m + bw, 0, 0, start, lvl});
  return start + bw - 1;
}
}  // namespace band_detail

// block steps (launches) of n blocks cut `depth` times; memo: of earlier calls
// with the same bandwidth
typedef std::map<std::pair<int, int>, std::pair<int, int>> StepMemo;
inline int band_steps(int n, int bw, int depth, StepMemo &memo) {
  return n <= 0 ? 0 : band_detail::last_level(n, bw > 0 ? depth : 0, bw, memo) + 1;
}
inline int band_steps(int n, int bw, int depth) {
  StepMemo memo;
  return band_steps(n, bw, depth, memo);
}

inline BandPlan make_band_plan(int n, int bw, bool sym, int depth) {
  using namespace band_detail;
  BandPlan P;
  P.n = n;
  P.bw = bw;
  P.sym = sym;
  if (n <= 0) return P;
  std::vector<Node> nodes;
  std::map<std::pair<int, int>, std::pair<int, int>> memo;
  const int nlev = cut(nodes, 0, n, bw > 0 ? depth : 0, bw, false, false, memo) + 1;
  const int nn = (int)nodes.size();
  std::vector<int> node_of(n), level(n), order;
  P.rank.assign(n, 0);
  P.leaves = 0;
  for (int v = 0; v < nn; ++v) {
    const Node &d = nodes[v];
    P.leaves += d.leaf;
    for (int q = 0; q < d.hi - d.lo; ++q) {
      const int b = d.desc ? d.hi - 1 - q : d.lo + q;
      node_of[b] = v;
      level[b] = d.start + q;
      P.rank[b] = (int)order.size();
      order.push_back(b);
    }
  }
  const std::vector<int> &rank = P.rank;
  std::vector<char> nz((size_t)n * n, 0), init((size_t)n * n, 0);
  for (int i = 0; i < n; ++i)
    for (int j = std::max(0, i - bw); j <= std::min(n - 1, i + bw); ++j) {
      nz[(size_t)i * n + j] = 1;
      if (!sym || rank[i] >= rank[j]) init[(size_t)i * n + j] = 1;
    }
  // pivots by level; column structures, and their rows (in elimination order of the columns)
  std::vector<std::vector<int>> at(nlev), st(n), pre(n);
  for (int b : order) at[level[b]].push_back(b);
  std::vector<int> slot((size_t)nn * n, -1);
  std::vector<char> written((size_t)nn * n, 0);
  auto slot_of = [&](int v, int i) -> int & { return slot[(size_t)v * n + i]; };
  // the blocks that the pivots of the level before update, and where a block's
  // target is (a table: a map of them took most of a plan's time)
  struct Target {
    int i, j, p0, p1, first;
  };
  std::vector<Target> tg;
  std::vector<int> where((size_t)n * n, -1);
  std::vector<std::vector<int>> by_node(nn);  // a level's other targets by the node of p0
  std::vector<int> active;                    // nodes of the level, ascending
  P.lev.resize(nlev);
  for (int l = 0; l < nlev; ++l) {
    BandPlan::Level &L = P.lev[l];
    static const std::vector<int> none;
    const std::vector<int> &pend = l > 0 ? at[l - 1] : none;
    tg.clear();
    for (int p : pend)
      for (int i : st[p])
        for (int j : st[p]) {
          if (sym && rank[i] < rank[j]) continue;
          int &w = where[(size_t)i * n + j];
          if (w < 0) {
            w = (int)tg.size();
            tg.push_back(Target{i, j, p, -1, init[(size_t)i * n + j] ? 0 : 1});
          } else if (tg[w].p1 < 0) {
            tg[w].p1 = p;
          } else {
            throw std::logic_error("band plan: three updates of one block in one launch");
          }
          ++L.products;
        }
    for (const Target &t : tg) init[(size_t)t.i * n + t.j] = 1;
    for (int s : at[l]) {
      for (int q = rank[s] + 1; q < n; ++q)
        if (nz[(size_t)s * n + order[q]]) st[s].push_back(order[q]);
      for (int i : st[s]) {
        pre[i].push_back(s);
        for (int j : st[s]) nz[(size_t)i * n + j] = 1;
      }
      BandPlan::Pivot pv{s, -1, (int)P.refs.size(), (int)st[s].size(), node_of[s]};
      const int d = where[(size_t)s * n + s];
      if (d >= 0) {
        if (tg[d].p1 >= 0) throw std::logic_error("band plan: two updates pending on a pivot");
        pv.p = tg[d].p0;
        tg[d].p0 = -1;  // taken
      }
      for (int i : st[s]) {
        BlockRef r{(int16_t)i, (int16_t)s, -1, -1, init[(size_t)i * n + s] ? 0 : 1, 0};
        const int e = where[(size_t)i * n + s];
        if (e >= 0) {
          if (tg[e].p1 >= 0 || tg[e].p0 != pv.p) throw std::logic_error("band plan: column updates differ");
          r.p0 = (int16_t)tg[e].p0;
          r.first = tg[e].first;
          tg[e].p0 = -1;
        }
        init[(size_t)i * n + s] = 1;
        if (!sym) init[(size_t)s * n + i] = 1;
        P.refs.push_back(r);
      }
      L.products += 1 + (long long)st[s].size();
      L.piv.push_back(pv);
    }
    std::vector<size_t> done;  // slots that this level writes: readable from the next one on
    // the other updated blocks, by the node whose pivot updates them first,
    // and the forward substitution of the nodes that are active
    active.clear();
    for (int s : at[l]) active.push_back(node_of[s]);
    for (int p : pend) active.push_back(node_of[p]);
    std::sort(active.begin(), active.end());
    active.erase(std::unique(active.begin(), active.end()), active.end());
    for (int v : active) by_node[v].clear();
    for (size_t k = 0; k < tg.size(); ++k) {
      where[(size_t)tg[k].i * n + tg[k].j] = -1;
      if (tg[k].p0 >= 0) by_node[node_of[tg[k].p0]].push_back((int)k);
    }
    for (int v : active) {
      BandPlan::Group g{(int)P.refs.size(), 0, (int)P.fops.size(), 0};
      std::sort(by_node[v].begin(), by_node[v].end(), [&](int a, int b) {
        return tg[a].i != tg[b].i ? tg[a].i < tg[b].i : tg[a].j < tg[b].j;
      });
      for (int k : by_node[v]) {
        const Target &t = tg[k];
        P.refs.push_back(BlockRef{(int16_t)t.i, (int16_t)t.j, (int16_t)t.p0, (int16_t)t.p1, t.first, 0});
      }
      auto op = [&](int kind, int i, int p, int sl) {
        P.fops.push_back(FwdOp{(int16_t)kind, (int16_t)i, (int16_t)p, 0, sl, 0});
      };
      for (int s : at[l]) {
        if (node_of[s] != v) continue;
        for (int t : pre[s])
          if (node_of[t] == v) op(FW_TERM, s, t, 0);
        for (int u = 0; u < nn; ++u)
          if (u != v && written[(size_t)u * n + s]) op(FW_SUB, s, 0, slot_of(u, s));
        for (int p : pend)
          if (node_of[p] != v && std::find(st[p].begin(), st[p].end(), s) != st[p].end()) op(FW_TERM, s, p, 0);
        op(FW_END, s, 0, 0);
      }
      for (int p : pend) {
        if (node_of[p] != v) continue;
        for (int i : st[p]) {
          if (node_of[i] == v || level[i] == l) continue;  // this level's pivot takes the product itself
          int &sl = slot_of(v, i);
          if (sl < 0) sl = P.nslot++;
          op(written[(size_t)v * n + i] ? FW_ACC : FW_ACC0, i, p, sl);
          done.push_back((size_t)v * n + i);
        }
      }
      g.nref = (int)P.refs.size() - g.ref0;
      g.nfop = (int)P.fops.size() - g.fop0;
      if (g.nref || g.nfop) L.grp.push_back(g);
    }
    for (size_t q : done) written[q] = 1;
    for (const BandPlan::Pivot &v : L.piv) BandPlan::count(L.pivs, v.nref, 0, 1);
    for (const BandPlan::Group &g : L.grp) BandPlan::count(L.grps, g.nref, g.nfop > 0, 1);
  }
  // ---- sweeps ----
  auto part = [&](SweepPart &S, int ops0, int loc0) {
    S.op0 = ops0;
    S.nop = (int)P.ops.size() - ops0;
    S.loc0 = loc0;
    S.nloc = (int)P.locs.size() - loc0;
  };
  std::vector<int> local(n, -1);
  auto add_loc = [&](int b, int init_kind, int out, int loc0) {
    local[b] = (int)P.locs.size() - loc0;
    SweepLoc q{};
    q.b = b;
    q.init = init_kind;
    q.out = out;
    q.acc0 = (int)P.accs.size();
    P.locs.push_back(q);
  };
  auto row = [&](int i, const std::vector<int> &cols, int end, int dst) {
    for (size_t q = 0; q < cols.size(); ++q)
      P.ops.push_back(SweepOp{(int16_t)i, (int16_t)cols[q], (int16_t)local[cols[q]],
                              (int16_t)(q + 1 == cols.size() ? end : SW_SUM), dst, 0});
  };
  auto leaf_of = [&](int b) { return nodes[node_of[b]].leaf ? node_of[b] : -1; };  // -1: the separators
  auto cols_of = [&](int i, int part_of) {  // the columns of row i in one leaf, or in the separators
    std::vector<int> cols;
    for (int t : pre[i])
      if (leaf_of(t) == part_of) cols.push_back(t);
    return cols;
  };
  auto fwd_rows = [&](const std::vector<int> &blocks) {
    for (int s : blocks) row(s, cols_of(s, leaf_of(s)), SW_FWD, local[s]);
  };
  auto bwd_rows = [&](const std::vector<int> &blocks) {
    for (size_t q = blocks.size(); q-- > 0;) {
      const int s = blocks[q];
      row(s, st[s], SW_BSUM, local[s]);
      P.ops.push_back(SweepOp{(int16_t)s, (int16_t)s, (int16_t)(st[s].empty() ? local[s] : -1), SW_DIAG, local[s], 1});
    }
  };
  std::vector<std::vector<int>> mine(nn);
  std::vector<int> top;
  for (int b : order) {
    mine[node_of[b]].push_back(b);
    if (!nodes[node_of[b]].leaf) top.push_back(b);
  }
  for (int v = 0; v < nn; ++v) {
    if (!nodes[v].leaf) continue;
    std::vector<int> ext;
    for (int t : mine[v])
      for (int i : st[t])
        if (node_of[i] != v && std::find(ext.begin(), ext.end(), i) == ext.end()) ext.push_back(i);
    SweepPart f, b;
    int o0 = (int)P.ops.size(), l0 = (int)P.locs.size();
    for (int t : mine[v]) add_loc(t, SL_RHS, SL_OUT_Y, l0);
    fwd_rows(mine[v]);
    for (int i : ext) {
      int &sl = slot_of(v, i);
      if (sl < 0) sl = P.nslot++;
      row(i, cols_of(i, v), SW_ACC, sl);
    }
    part(f, o0, l0);
    P.fwd.push_back(f);
    o0 = (int)P.ops.size();
    l0 = (int)P.locs.size();
    for (int t : mine[v]) add_loc(t, SL_Y, SL_OUT_D, l0);
    for (int i : ext) add_loc(i, SL_X, 0, l0);
    bwd_rows(mine[v]);
    part(b, o0, l0);
    P.bwd.push_back(b);
  }
  // separator by separator, the deepest first
  int depth_of = 0, nsep = 0;
  for (const Node &d : nodes)
    if (!d.leaf) {
      depth_of = std::max(depth_of, d.lvl);
      ++nsep;
    }
  if (nsep >= 3) {
    P.sep_fwd.resize(depth_of + 1);
    P.sep_bwd.resize(depth_of + 1);
    std::vector<std::vector<int>> exts(nn);
    for (int v = 0; v < nn; ++v)
      for (int t : mine[v])
        for (int i : st[t])
          if (node_of[i] != v && std::find(exts[v].begin(), exts[v].end(), i) == exts[v].end()) exts[v].push_back(i);
    auto own_cols = [&](int i, int v) {
      std::vector<int> cols;
      for (int t : pre[i])
        if (node_of[t] == v) cols.push_back(t);
      return cols;
    };
    for (int lvl = depth_of; lvl >= 0; --lvl)
      for (int v = 0; v < nn; ++v) {
        if (nodes[v].leaf || nodes[v].lvl != lvl) continue;
        // forward: the right-hand side minus what every part below left for its rows
        int o0 = (int)P.ops.size(), l0 = (int)P.locs.size();
        for (int b : mine[v]) {
          add_loc(b, SL_RHS, lvl == 0 ? SL_OUT_Y | SL_OUT_D : SL_OUT_Y, l0);
          for (int u = 0; u < nn; ++u)
            if (u != v && std::find(exts[u].begin(), exts[u].end(), b) != exts[u].end()) {
              P.accs.push_back(slot_of(u, b));
              ++P.locs.back().nacc;
            }
        }
        for (int b : mine[v]) row(b, own_cols(b, v), SW_FWD, local[b]);
        if (lvl == 0) {
          const int o1 = (int)P.ops.size();
          bwd_rows(mine[v]);
          part(P.root, o0, l0);
          part(P.root_bwd, o1, l0);
          continue;
        }
        for (int i : exts[v]) {
          int &sl = slot_of(v, i);
          if (sl < 0) sl = P.nslot++;
          row(i, own_cols(i, v), SW_ACC, sl);
        }
        SweepPart f, b;
        part(f, o0, l0);
        P.sep_fwd[lvl].push_back(f);
        o0 = (int)P.ops.size();
        l0 = (int)P.locs.size();
        for (int t : mine[v]) add_loc(t, SL_Y, SL_OUT_Y | SL_OUT_D, l0);
        for (int i : exts[v]) add_loc(i, SL_X, 0, l0);
        bwd_rows(mine[v]);
        part(b, o0, l0);
        P.sep_bwd[lvl].push_back(b);
      }
  }
  {
    const int o0 = (int)P.ops.size(), l0 = (int)P.locs.size();
    for (int b : order) add_loc(b, SL_RHS, SL_OUT_D, l0);
    for (int s : order) row(s, pre[s], SW_FWD, local[s]);
    const int o1 = (int)P.ops.size();
    bwd_rows(order);
    part(P.whole, o0, l0);
    part(P.whole_bwd, o1, l0);
  }
  if (!top.empty()) {
    const int l0 = (int)P.locs.size();
    for (int b : top) {
      add_loc(b, SL_RHS, SL_OUT_Y | SL_OUT_D, l0);
      for (int v = 0; v < nn; ++v)
        if (nodes[v].leaf && slot_of(v, b) >= 0) {
          P.accs.push_back(slot_of(v, b));
          ++P.locs.back().nacc;
        }
    }
    const int o0 = (int)P.ops.size();
    fwd_rows(top);
    const int o1 = (int)P.ops.size();
    bwd_rows(top);
    part(P.top, o0, l0);
    part(P.top_bwd, o1, l0);
  }
  return P;
}

}  // namespace wcfe
