"""What a context refuses, and the device memory that it takes and gives back."""
import ctypes
import threading
import time

import numpy as np
import pytest

import cells
from wholecellfe_amd import mesh

pytestmark = pytest.mark.gpu

W = pytest.importorskip("wholecellfe_amd")


def free_bytes():
    """Free device memory, from the HIP runtime that the library is linked to."""
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert W.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def most_free(seconds=0.5):
    """The runtime gives memory back some time after the call that frees it."""
    end, most = time.monotonic() + seconds, 0
    while time.monotonic() < end:
        most = max(most, free_bytes())
        time.sleep(0.01)
    return most


# a checkpoint holds at most 2047 cells, and the LU's work lists 11 bits of them
def test_batches_above_2047_cells_are_refused():
    X, T, _ = mesh.disk_rings(1, 10.0)
    for n in (2047, 2048):
        with W.Context(t0=1.0) as c:
            for _ in range(n):
                c.add_cell(X=X, tris=T, law=W.LAW_CST, E=1000.0, spr_tri=np.zeros(1, np.int32),
                           spr_bary=np.full((1, 3), 1 / 3), spr_anchor=X[T[0]].mean(axis=0)[None])
            if n < 2048:
                c.finalize()
                continue
            with pytest.raises(W.WcfeError) as e:
                c.finalize()
            assert e.value.code == W.ERR_ARG


def solve(c, n, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) / np.sqrt(n) + 3.0 * np.eye(n)
    b = rng.standard_normal(n)
    return A, b, c.dense_solve([A], [b])[0][0]


# A (FP64), the factors (FP64) and 128 entries per row of diagonal inverses
def test_large_dense_solve_takes_what_it_needs():
    n = 6000
    need = 8 * (n * n + 6016 * 6016 + 128 * 6016)
    with W.Context(precision=W.PREC_FP64) as c:
        solve(c, 200, 1)  # code and streams are loaded
        before, least, stop = most_free(), [1 << 62], threading.Event()

        def watch():
            while not stop.is_set():
                least[0] = min(least[0], free_bytes())

        t = threading.Thread(target=watch)
        t.start()
        try:
            A, b, x = solve(c, n, 2)
        finally:
            stop.set()
            t.join()
        after = most_free()
    used = before - least[0]
    print("needed %d, taken %d, kept %d" % (need, used, before - after), flush=True)
    assert np.linalg.norm(A @ x - b) <= 1e-8 * np.linalg.norm(b)
    assert 0.9 * need < used <= 1.1 * need  # vectors and 2 MiB granules beside the matrices
    assert before - after <= 64 << 20


# each thread's calls are its own, whichever holds the context's buffers
def test_two_threads_in_one_context():
    with W.Context(precision=W.PREC_FP64) as c:
        bad = []

        def work(seed):
            for k in range(12):
                A, b, x = solve(c, 40 + 90 * ((seed + k) % 4), 100 * seed + k)
                if not np.linalg.norm(A @ x - b) <= 1e-8 * np.linalg.norm(b):
                    bad.append((seed, k))

        ts = [threading.Thread(target=work, args=(s,)) for s in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    assert not bad


# two concurrent cell groups: the captured step runs on streams of its own
@pytest.mark.parametrize("groups", [0, 2])
def test_closed_contexts_give_their_memory_back(groups):
    ds = [cells.cst_cell(K=28, n_spr=100, seed=k, time=1.0) for k in range(4)]

    def one():
        with W.Context(t0=1.0, lu_groups=groups) as c:
            for d in ds * 4:
                cells.add_to_context(c, d)
            c.finalize()
            c.newton_step()
            return free_bytes()

    one()
    before = most_free()
    inside = [one() for _ in range(3)]
    # 16 cells of 4704 elements: 16 x 4872^2 x 4 bytes of matrices
    assert before - max(inside) > 1.4e9
    assert before - most_free() <= 64 << 20


# the autotuner lays the batch out many times, with other matrices and without
def test_autotuned_contexts_give_their_memory_back():
    d = cells.cst_cell(K=34, n_spr=100, seed=1, time=1.0)

    def one():
        with W.Context(t0=1.0) as c:
            for _ in range(8):
                cells.add_to_context(c, d)
            c.finalize()
            inside = free_bytes()
            c.autotune(steps=1)
            return inside

    one()
    before = most_free()
    inside = one()
    # 8 cells of 6936 elements: 8 x 7142^2 x 4 bytes of matrices
    assert before - inside > 1.5e9
    assert before - most_free() <= 64 << 20
