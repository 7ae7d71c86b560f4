"""Partial-pivoting panels and row interchanges at the edges of their forms:
rows per thread (512, 1024, 2048 rows), 64-row remainders, one column left.

The pivots equal LAPACK's on random systems (their column maxima differ far
more than rounding), for which FP64 refinement is converged: the relative
residual of the solution is within n eps of the backward-stable bound."""
import numpy as np
import pytest
from scipy.linalg import lu_factor

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


@pytest.mark.parametrize("n", [1, 17, 64, 65, 129, 500, 513, 640, 1025, 2049])
def test_pivots_equal_lapack(n):
    print("case n", n, flush=True)
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    b = rng.standard_normal(n)
    with W.Context(precision=W.PREC_FP64, pivoting=W.PIVOT_PARTIAL) as c:
        xs, rel, _, piv = c.dense_solve([A, A[: (n + 1) // 2, : (n + 1) // 2]], [b, b[: (n + 1) // 2]])
    assert np.array_equal(piv[:n], lu_factor(A)[1])
    assert np.array_equal(piv[n:], lu_factor(A[: (n + 1) // 2, : (n + 1) // 2])[1])
    eps = np.finfo(float).eps
    assert np.linalg.norm(b - A @ xs[0]) <= 8 * n * eps * np.linalg.norm(A) * np.linalg.norm(xs[0])


def test_mixed_precision_pivots_and_residual():
    rng = np.random.default_rng(3)
    sizes = [40, 511, 600, 1100]
    mats = [rng.standard_normal((n, n)) + 2 * np.sqrt(n) * np.diag(rng.choice([-1.0, 1.0], n)) for n in sizes]
    rhss = [rng.standard_normal(n) for n in sizes]
    with W.Context(precision=W.PREC_MIXED, pivoting=W.PIVOT_PARTIAL) as c:
        xs, rel, _, piv = c.dense_solve(mats, rhss)
    o = 0
    for A, b, x, n in zip(mats, rhss, xs, sizes):
        assert np.linalg.norm(b - A @ x) <= 1e-8 * np.linalg.norm(b)
        assert np.array_equal(piv[o:o + n], lu_factor(A.astype(np.float32))[1])
        o += n
