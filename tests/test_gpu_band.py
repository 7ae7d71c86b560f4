"""The band LU with its cuts, FP32 and FP64, on single cells from one block to
about thirty (one leaf, two, and several), symmetric and not: the Newton step
solves the oracle's system."""
import numpy as np
import pytest

import cells
import oracle_py as O

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


# rings K: 6 K^2 triangles, 3 K (K + 1) + 1 nodes
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
@pytest.mark.parametrize("sym", [1, 0])
@pytest.mark.parametrize("K", [1, 2, 4, 6, 8, 11, 17])
def test_newton_step_solves_the_oracle_system(K, sym, prec):
    print("case K", K, "sym", sym, "prec", prec, flush=True)
    d = cells.cst_cell(K=K, n_spr=10 * K, law_table=K % 2 == 0, seed=K, time=1.0)
    G, Kd = O.assemble(O.make_cell(d))
    for twist in (1, 0):
        with W.Context(precision=prec, t0=1.0, symmetric=sym, twist=twist, max_refine=8) as c:
            cells.add_to_context(c, d)
            c.finalize()
            st = c.newton_step()
            dx = c.positions(0) - d["x"]
        # lin_rtol is 1e-8 on the GPU's own assembled system, which equals the oracle's to 1e-12
        assert st["max_lin_relres"] <= 1e-8
        assert np.linalg.norm(-G - Kd @ dx) <= 1.1e-8 * np.linalg.norm(G)
        if prec == W.PREC_FP64:
            # one FP64 solve of a system of condition below 1e6: far below lin_rtol without refinement
            assert st["max_refine_used"] == 1 and st["max_lin_relres"] <= 1e-10
