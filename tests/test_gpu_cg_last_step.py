"""The last step of the FP64 CG reaches every row (csrc/ngpb_krylov.hip, k_pcg_dir).

The launch that raises the stop flag also adds the last alpha p to x, so no block of it may
be turned away by that flag. Other contexts solve on their own streams meanwhile, which
delays the start of blocks. With one iteration the last step is the whole solution,
x = alpha D^-1 b; a converged solve is the same bit for bit as alone, and the residual it
reports is that of the x it returns.
"""
import ctypes
import threading
from contextlib import contextmanager

import numpy as np
import pytest
import scipy.sparse as sp

from cudanextgenpb_amd import native

from test_zz_no_alloc import DeviceArray, hip

pytestmark = pytest.mark.gpu


def grid_system(m, seed):
    """Seven-point operator with varying coefficients on m^3 nodes, and a full right-hand side."""
    rng = np.random.default_rng(seed)
    n = m**3
    i = np.arange(n)
    pairs = []
    for step, pos in ((1, i % m), (m, i // m % m), (m * m, i // (m * m))):
        a = i[pos < m - 1]
        pairs.append(np.stack([a, a + step], 1))
    pairs = np.concatenate(pairs)
    A = sp.coo_matrix((-rng.uniform(0.5, 1.5, len(pairs)), (pairs[:, 0], pairs[:, 1])), shape=(n, n)).tocsr()
    A = A + A.T
    A = (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.05)).tocsr()
    A.sort_indices()
    return A, rng.uniform(0.5, 1.5, n) * rng.choice([-1.0, 1.0], n)


@contextmanager
def busy_device(threads=3):
    """Solves on `threads` other contexts until the block ends."""
    stop, failed = threading.Event(), []

    def work(k):
        try:
            A, b = grid_system(40 + 8 * k, 100 + k)
            with native.Context(0) as c:
                c.set_csr(A.indptr, A.indices, A.data, b)
                while not stop.is_set():
                    c.solve(native.PREC_FP64 if k % 2 else native.PREC_MIXED, tol=1e-10)
        except Exception as e:  # pragma: no cover
            failed.append(e)

    pool = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in pool:
        t.start()
    try:
        yield
    finally:
        stop.set()
        for t in pool:
            t.join()
    assert not failed, failed


def solve_noalloc(h, A, b, tol, maxiter):
    arrs = [DeviceArray(h, a) for a in (A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, b,
                                        np.full(len(b), np.nan))]
    o = native.SolveOpts(native.PREC_FP64, tol, maxiter, 1e-3, 8, native.SOLVER_CG, native.PRECON_JACOBI, 1.0)
    st = native.SolveStats()
    native.lib().ngpb_solve_csr_noalloc(0, None, len(b), len(A.data), *[a.p for a in arrs], ctypes.byref(o),
                                        ctypes.byref(st))
    x = arrs[4].get()
    for a in arrs:
        a.free()
    return x, st.as_dict()


def solve_context(A, b, tol, maxiter):
    with native.Context(0) as c:
        c.set_csr(A.indptr, A.indices, A.data, b)
        return c.solve(native.PREC_FP64, tol=tol, maxiter=maxiter, check_every=8, raise_on_noconv=False)


@pytest.mark.parametrize("m", [17, 40, 100])  # just above the one-block solver, one row per thread, four
def test_one_iteration_reaches_every_row(m):
    A, b = grid_system(m, m)
    p = (1.0 / A.diagonal()) * b  # the first direction, as the solver forms it
    h = hip()
    with busy_device():
        for r in range(4):
            print(f"[last step] {m}^3 rows, one iteration, pass {r}", flush=True)
            for x, st in (solve_context(A, b, 1e-10, 1), solve_noalloc(h, A, b, 1e-10, 1)):
                assert st["iterations"] == 1 and st["status"] == 4
                alpha = x / p
                # x and the division round once each
                assert np.all(np.abs(alpha - np.median(alpha)) <= 4 * np.finfo(float).eps * np.median(alpha))


def test_solves_beside_others_are_the_same():
    A, b = grid_system(60, 1)
    h = hip()
    alone = solve_context(A, b, 1e-8, 10000)
    alone_na = solve_noalloc(h, A, b, 1e-8, 10000)
    with busy_device():
        for r in range(5):
            print(f"[last step] 60^3 rows beside others, pass {r}", flush=True)
            for ref, got in ((alone, solve_context(A, b, 1e-8, 10000)), (alone_na, solve_noalloc(h, A, b, 1e-8, 10000))):
                x, st = got
                assert st["status"] == 0 and st["iterations"] == ref[1]["iterations"]
                true = np.linalg.norm(A @ x - b) / np.linalg.norm(b)
                # the recursive residual drifts by rounding, some 1e-13 of ||b|| here
                assert abs(true - st["relres"]) <= 1e-4 * st["relres"], (true, st["relres"])
                assert np.array_equal(x, ref[0]), (np.sum(x != ref[0]), np.abs(x - ref[0]).max())
