"""A cell's Newton steps do not depend on the batch it is in: alone, one
workgroup runs its refinement and ends its step; beside enough other cells the
same phases run as batch-wide launches, with one workgroup per cell only for
the sweeps after the second."""
import numpy as np
import pytest

import cells

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


def states(ds, prec, lin_rtol, kinetics, n):
    with W.Context(precision=prec, t0=1.0, lin_rtol=lin_rtol, max_refine=5) as c:
        for d in ds:
            cells.add_to_context(c, d, kinetics=kinetics)
        c.finalize()
        for _ in range(4):
            c.newton_step(stats=False)
        c.synchronize()
        return [(c.positions(i),) + tuple(c.ul_state(i)) for i in range(n)]


# lin_rtol 0: all five sweeps run
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
@pytest.mark.parametrize("lin_rtol", [1e-12, 0.0])
@pytest.mark.parametrize("kind", ["spring", "ul"])
def test_cell_alone_equals_cell_in_a_large_batch(kind, lin_rtol, prec):
    print("case", kind, lin_rtol, prec, flush=True)
    make = (lambda K: cells.cst_cell(K=K, n_spr=10 * K, seed=K, time=1.0)) if kind == "spring" else \
        (lambda K: cells.ul_cell(K=K, seed=K))
    kin = 0 if kind == "spring" else W.KIN_MEANFIELD
    few = [make(K) for K in (1, 2, 5)]
    # 10 disks of 6936 triangles: above 65536 elements, and too long for one workgroup's whole refinement
    filler = [make(34) for _ in range(10)]
    lone = [states([d], prec, lin_rtol, kin, 1)[0] for d in few]
    many = states(few + filler, prec, lin_rtol, kin, len(few))
    for d, a, b in zip(few, lone, many):
        move = np.linalg.norm(b[0] - np.asarray(d["x"]).ravel())
        # relative residual 1e-12 at a condition number below 1e6
        assert np.linalg.norm(a[0] - b[0]) <= 1e-6 * move
        for p, q in zip(a[1:], b[1:]):
            assert np.abs(p - q).max() <= 1e-6 * max(1.0, np.abs(q).max())


# K = 1: one block (no band); 2 and more: the band with the area term's rank
# one added by Sherman-Morrison, against the full matrix with row pivoting
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
@pytest.mark.parametrize("K", [1, 2, 5, 11])
def test_area_term_in_the_band_equals_the_full_matrix(K, prec):
    print("case area", K, prec, flush=True)
    d = cells.ul_cell(K=K, seed=K)
    out = []
    for piv in (W.PIVOT_STATIC, W.PIVOT_PARTIAL):
        with W.Context(precision=prec, t0=1.0, lin_rtol=1e-12, max_refine=8, pivoting=piv) as c:
            c.set_table(0, d["tab_px"], d["tab_py"], d["tab_k"])
            c.add_cell(X=d["X"], x=d["x"], tris=d["tris"], law=d["law"], mu=d["mu"], thick=d["thick"], ea=d["ea"],
                       node_springs=1, cC=d["cC"], fau=d["fau0"], rho_max=d["rho_max"], spring_law=1,
                       kinetics=W.KIN_MEANFIELD, k_bend=W.K_BEND_REF, k_area=W.K_AREA_REF, drag=W.DRAG_REF)
            c.finalize()
            Kmat = c.assembled_system(0)[0]
            for _ in range(3):
                c.newton_step(stats=False)
            c.synchronize()
            out.append((c.positions(0), Kmat))
    (xs, Ks), (xf, Kf) = out
    assert np.abs(Ks - Kf).max() <= 1e-12 * np.abs(Kf).max()  # the same sums, rounded alike
    # relative residual 1e-12 at a condition number below 1e6
    assert np.linalg.norm(xs - xf) <= 1e-6 * np.linalg.norm(xf - np.asarray(d["x"]).ravel())


# 7994 and 8438 unknowns: one and two partial sums of the norms
@pytest.mark.parametrize("K", [36, 37])
def test_norms_of_large_cells(K):
    print("case norm", K, flush=True)
    d = cells.cst_cell(K=K, n_spr=500, seed=K, time=1.0)
    # tolerances of zero: the load step stays open, its residual at time t0
    with W.Context(t0=1.0, newton_rtol=0.0, newton_atol=0.0) as c:
        cells.add_to_context(c, d)
        c.finalize()
        g0 = np.linalg.norm(c.residual(0))
        st = c.newton_step()
        g1 = np.linalg.norm(c.residual(0))
    # 8438 rounded squares, and the residual summed in another order
    assert abs(st["max_newton_rel"] - g1 / g0) <= 1e-9 * (g1 / g0) + 1e-15


# 9600 and 15000 elements alone: a band cut deep enough that the separators are
# swept by depth, against the uncut band
@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
@pytest.mark.parametrize("sym", [1, 0])
@pytest.mark.parametrize("K", [40, 50])
def test_separators_by_depth_equal_the_uncut_band(K, sym, prec):
    print("case depth", K, sym, prec, flush=True)
    d = cells.cst_cell(K=K, n_spr=400, seed=K, time=1.0)
    out = []
    for twist in (1, 0):
        with W.Context(precision=prec, t0=1.0, symmetric=sym, twist=twist, lin_rtol=1e-12, max_refine=8) as c:
            cells.add_to_context(c, d)
            c.finalize()
            c.newton_step()
            out.append(c.positions(0))
    # relative residual 1e-12 at a condition number below 1e6
    assert np.linalg.norm(out[0] - out[1]) <= 1e-6 * np.linalg.norm(out[1] - d["x"])


# The first FP32 solve, whose forward substitution ran beside the
# factorization: a sweep that reads the wrong vector leaves the residual at 1
@pytest.mark.parametrize("sym", [1, 0])
@pytest.mark.parametrize("K", [1, 4, 11, 17, 40])
def test_first_solve_reduces_the_residual(K, sym):
    print("case first solve", K, sym, flush=True)
    d = cells.cst_cell(K=K, n_spr=10 * K, seed=K, time=1.0)
    with W.Context(precision=W.PREC_MIXED, t0=1.0, symmetric=sym, max_refine=1, lin_rtol=0.1) as c:
        cells.add_to_context(c, d)
        c.finalize()
        # FP32 roundoff 6e-8 times a condition number below 1e6
        assert c.newton_step()["max_lin_relres"] <= 0.1
