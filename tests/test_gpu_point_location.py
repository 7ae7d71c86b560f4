"""The explicit calls' point location, one wave per node: candidate lists of one
to several wavefronts, nodes in one to three triangles (the last two come back
separately from the third on), against the oracle."""
import numpy as np
import pytest

import oracle_py as O
from wholecellfe_amd import mesh

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


def substrate(side, layers, planar):
    """`layers` copies of a grid of 2 side^2 triangles; a node a little off the
    plane puts every triangle in every point's candidate list."""
    X, T = mesh.substrate_grid(side, 20.0)
    n = len(X)
    X = np.concatenate([np.concatenate([X, np.zeros((n, 1))], axis=1)] * layers)
    T = np.concatenate([T + k * n for k in range(layers)])
    if not planar:
        X = np.concatenate([X, [[0.0, 0.0, 1.0]]])
    return X, T


@pytest.mark.parametrize("side,layers,planar", [(2, 1, True), (4, 2, False), (6, 3, False), (8, 3, True)])
@pytest.mark.parametrize("law", [0, 1])
def test_point_location_against_the_oracle(side, layers, planar, law):
    print("case", side, layers, planar, law, flush=True)
    rng = np.random.default_rng(side)
    C, CT, _ = mesh.disk_rings(5, 10.0)
    n = len(C)
    X = np.concatenate([C, np.zeros((n, 1))], axis=1)
    x = X + np.concatenate([0.01 * rng.standard_normal((n, 2)), np.zeros((n, 1))], axis=1)
    fau = np.concatenate([0.004 * rng.standard_normal((n, 2)), np.zeros((n, 1))], axis=1)
    cA, cC = np.full(n, 100.0), rng.uniform(0.2, 1.0, n)
    SX, ST = substrate(side, layers, planar)
    Sx = SX + np.concatenate([0.001 * rng.standard_normal((len(SX), 2)), np.zeros((len(SX), 1))], axis=1)
    with W.Context() as c:
        a = c.update_fa(X.reshape(-1), x.reshape(-1), cA, cC, fau.reshape(-1), 0.005, ST.reshape(-1), SX.reshape(-1),
                        Sx.reshape(-1), law, 1000.0)
        F = c.force_fa_subs(CT.reshape(-1), x.reshape(-1), cC, fau.reshape(-1), ST.reshape(-1), Sx.reshape(-1), law,
                            1000.0)
    o = O.update_fa(CT, X, x, cA, cC, fau, 0.005, ST, SX, Sx, law, 1000.0)
    Fo = O.force_fa_subs(CT, x, cC, fau, ST, Sx, law, 1000.0)
    assert a[3] == o[3]
    # the same operations in the same order, FP64 without contraction
    for p, q in zip(a[:3], o[:3]):
        assert np.abs(np.ravel(p) - np.ravel(q)).max() <= 1e-13 * max(1.0, np.abs(q).max())
    assert np.abs(F - Fo).max() <= 1e-13 * np.abs(Fo).max()
