"""Small cells of the reference's whole model (bending, drag, actin
polymerisation, one with the area term) alone and beside enough other cells
that the step's phases run as batch-wide launches: the same states.  The area
cell's refinement runs in one workgroup beside cells that are swept by
launches."""
import numpy as np
import pytest

import cells

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


def small(K, area):
    d = cells.ul_cell(K=K, seed=K, table=False)
    d["terms"] = dict(k_bend=W.K_BEND_REF, k_area=W.K_AREA_REF if area else 0.0, drag=W.DRAG_REF, ap=0 if area else 1)
    return d


def states(ds, prec, n, steps):
    with W.Context(precision=prec, t0=1.0, dt=0.005, lin_rtol=1e-12, max_refine=6, newton_rtol=1e-10,
                   newton_atol=1e-8) as c:
        for d in ds:
            c.add_cell(X=d["X"], x=d["x"], tris=d["tris"], law=d["law"], mu=d["mu"], thick=d["thick"], ea=d["ea"],
                       node_springs=1, cC=d["cC"], fau=d["fau0"], rho_max=d["rho_max"], spring_law=0,
                       k_lin=d["k_lin"], kinetics=W.KIN_MEANFIELD, **d.get("terms", {}))
        c.finalize()
        layout = [c.cell_layout(i) for i in range(n)]
        for _ in range(steps):
            c.newton_step(stats=False)
        c.synchronize()
        info = [c.cell_info(i) for i in range(n)]
        return [(c.positions(i),) + tuple(c.ul_state(i)) for i in range(n)], info, layout


@pytest.mark.parametrize("prec", [W.PREC_MIXED, W.PREC_FP64])
def test_boundary_terms_in_a_large_batch(prec):
    print("case", prec, flush=True)
    # the actin draws are the cell's own (stream 0): one cell with them, first in both batches
    few = [small(5, False), small(4, True), small(7, True)]
    few[2]["terms"]["ap"] = 0
    # 10 disks of 6936 triangles: above 65536 elements, too long for one workgroup's whole refinement
    filler = [cells.ul_cell(K=34, seed=34, table=False) for _ in range(10)]
    lone = [states([few[0]], prec, 1, 5)] + [states([d], prec, 1, 5) for d in few[1:]]
    many, info, layout = states(few + filler, prec, len(few), 5)
    for i, d in enumerate(few):
        (a,), (ia,), (la,) = lone[i]
        b = many[i]
        assert la["bw"] == layout[i]["bw"] < la["nblk"] - 1 or la["nblk"] <= 3  # the band, also of the area cells
        assert ia["step"] == info[i]["step"] >= 1
        move = np.linalg.norm(b[0] - np.asarray(d["x"]).ravel())
        # relative residual 1e-12 at a condition number below 1e6
        assert np.linalg.norm(a[0] - b[0]) <= 1e-6 * move
        for p, q in zip(a[1:], b[1:]):
            assert np.abs(p - q).max() <= 1e-6 * max(1.0, np.abs(q).max())
