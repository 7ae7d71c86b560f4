"""The reported cuts are those of the plan that runs."""
import pytest

import cells

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


def layouts(ds, **opt):
    with W.Context(t0=1.0, **opt) as c:
        for d in ds:
            cells.add_to_context(c, d)
        c.finalize()
        return [c.cell_layout(i) for i in range(len(ds))]


@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
def test_reported_cuts(prec):
    ds = [cells.cst_cell(K=k, n_spr=20 + 10 * k, seed=k, time=1.0) for k in (3, 9, 16, 27)]
    for l in layouts(ds, precision=prec, twist=0):
        assert l["leaves"] == 1 and l["levels"] == l["nblk"]
    for l in layouts(ds, precision=prec, twist=2):  # at most one cut
        assert l["leaves"] in (1, 2)
        # both sides take half the blocks off the separator, one block step each, then the separator
        if l["leaves"] == 2:
            half = (l["nblk"] - l["bw"] + 1) // 2
            assert half + l["bw"] <= l["levels"] <= half + l["bw"] + 2
    alone = layouts(ds[-1:], precision=prec)[0]  # one latency-bound chain: several cuts
    assert alone["leaves"] > 2 and alone["levels"] < alone["nblk"] // 2
    assert alone["chain_top"] > 0
    sparse = layouts([ds[0]], precision=prec, dense_max_dof=0)[0]
    assert sparse["solver"] == W.SOLVER_CSR and sparse["leaves"] == 0 and sparse["levels"] == 0


# one cell of 5400 elements whose band starts uncut: cut it takes about half
# the time, in either precision
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
def test_autotune_tries_the_cuts(prec):
    d = cells.cst_cell(K=30, n_spr=300, seed=1, time=1.0)
    with W.Context(t0=1.0, precision=prec, twist=0, lu_depth=1, lu_groups=1) as c:
        cells.add_to_context(c, d)
        c.finalize()
        assert c.cell_layout(0)["leaves"] == 1
        ch = c.autotune(W.TUNE_LU, steps=2)
        print(ch, c.cell_layout(0), flush=True)
        assert ch["fused_step"] > 0 and c.cell_layout(0)["leaves"] > 2
