"""Cells with the area term, factored as a band matrix B = K - k g g^T and a
rank one (g = dA/dx): area stiffnesses where the rank one decides the
solution, and areas off area_0 at which B is singular while K is not.  Both
against the oracle's FP64 system."""
import numpy as np
import pytest
import scipy.linalg as sl

import cells
import oracle_py as O

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


def area_cell(K, k_area):
    d = cells.ul_cell(K=K, seed=K, table=False)
    d.update(k_bend=W.K_BEND_REF, k_area=k_area, drag=W.DRAG_REF, dt=0.005)
    p = d["x"].reshape(-1, 2)[d["tris"].reshape(-1, 3)]
    d["area_0"] = 0.5 * np.abs((p[:, 1, 0] - p[:, 0, 0]) * (p[:, 2, 1] - p[:, 0, 1]) -
                               (p[:, 1, 1] - p[:, 0, 1]) * (p[:, 2, 0] - p[:, 0, 0])).sum()
    return d


def system(d, **over):
    return O.assemble(O.make_cell(dict(d, **over)))


def step(d, prec, max_refine):
    """One Newton step: the update and its statistics."""
    with W.Context(precision=prec, t0=d["time"], dt=d["dt"], lin_rtol=1e-8, max_refine=max_refine) as c:
        c.add_cell(X=d["X"], x=d["x"], tris=d["tris"], law=d["law"], mu=d["mu"], thick=d["thick"], ea=d["ea"],
                   node_springs=1, cC=d["cC"], fau=d["fau0"], rho_max=d["rho_max"], spring_law=0, k_lin=d["k_lin"],
                   k_bend=d["k_bend"], k_area=d["k_area"], area_0=d["area_0"], drag=d["drag"])
        c.finalize()
        st = c.newton_step(check=False)
        return c.positions(0) - d["x"], st


def check(d, dx, st):
    # lin_rtol is 1e-8 on the GPU's own system, which equals the oracle's to 1e-12
    G, K = system(d)
    print("sweeps", st["max_refine_used"], "relres", st["max_lin_relres"], flush=True)
    # far off area_0 a full Newton step may turn an element over: not the solve's matter
    assert st["error"] in (W.OK, W.ERR_DEGENERATE) and st["max_lin_relres"] <= 1e-8
    assert np.linalg.norm(-G - K @ dx) <= 1.1e-8 * np.linalg.norm(G)


# k g.B^-1 g from 13 to 1e7: without the rank one, or with z = B^-1 k g to FP32
# only, the residual does not fall; with it each sweep leaves FP32 roundoff
# (6e-8) times a condition number below 1e4
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
@pytest.mark.parametrize("k_area", [1e4, 1e6, 1e8])
@pytest.mark.parametrize("K", [3, 6, 11])
def test_stiff_area_term(K, k_area, prec):
    print("case stiff", K, k_area, prec, flush=True)
    d = area_cell(K, k_area)
    d["area_0"] *= 1.0 + 1e-3 / k_area
    dx, st = step(d, prec, 4)
    check(d, dx, st)
    assert st["max_refine_used"] <= 3


# B = C + (area_0 - A) H is linear in area_0: at the generalized eigenvalues of
# (C, -H) it is singular, and K is not (condition 2e3 to 4e5)
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
@pytest.mark.parametrize("which", ["first", "second", "negative"])
@pytest.mark.parametrize("K,k_area", [(3, 1e4), (6, 1e2), (6, 1e4), (9, 1e4), (11, 1e4)])
def test_band_part_singular(K, k_area, which, prec):
    print("case singular", K, k_area, which, prec, flush=True)
    d = area_cell(K, k_area)
    A = d["area_0"]
    C = system(d, k_area=0.0)[1]
    gg = system(d)[1] - C
    H = (system(d, area_0=A + 1.0)[1] - gg - C)
    w = sl.eig(C, -H, right=False)
    w = w[np.isfinite(w)]
    w = w[np.abs(w.imag) < 1e-9 * np.abs(w)].real
    shift = {"first": np.sort(w[w > 0])[0], "second": np.sort(w[w > 0])[1], "negative": np.sort(w[w < 0])[-1]}[which]
    d["area_0"] = A + shift
    sv = np.linalg.svd(C + shift * H, compute_uv=False)
    assert sv[-1] < 1e-10 * sv[0]
    dx, st = step(d, prec, 4)
    check(d, dx, st)


# max_refine holds where the sweeps converge: one sweep of an ordinary cell
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
def test_one_sweep_stays_one(prec):
    print("case one sweep", prec, flush=True)
    d = area_cell(6, W.K_AREA_REF)
    with W.Context(precision=prec, t0=d["time"], dt=d["dt"], lin_rtol=1e-14 if prec else 1e-12, max_refine=1) as c:
        c.add_cell(X=d["X"], x=d["x"], tris=d["tris"], law=d["law"], mu=d["mu"], thick=d["thick"], ea=d["ea"],
                   node_springs=1, cC=d["cC"], fau=d["fau0"], rho_max=d["rho_max"], spring_law=0, k_lin=d["k_lin"],
                   k_bend=d["k_bend"], k_area=d["k_area"], area_0=d["area_0"], drag=d["drag"])
        c.finalize()
        assert c.newton_step(check=False)["max_refine_used"] == 1
