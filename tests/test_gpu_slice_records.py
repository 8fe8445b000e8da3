"""FP64 CG on CSR systems whose 64-row slices take each form of the slice records.

Strictly diagonally dominant symmetric systems (condition number below 3) solved to a
relative residual of 1e-13 by ngpb_solve_csr_noalloc: the relative error is then below
3e-13 plus rounding. Sizes lie around the slice (64) and block (256) edges; the entries
lie on few diagonals with one value each, on few diagonals with varying values, on
exactly as many diagonals as a record holds and one more, or anywhere. Up to 4,096 rows, on
at most 14 diagonals (nine a slice on average at 4,096 rows), one block runs the whole CG
with 1, 2 or 4 rows per thread, 1,024 iterations per launch. Systems with slices that have no record are multiplied from the
CSR up to 2^18 rows and where most slices are such; the largest sizes here have a third
of them, around the rows from which records are used, and several staged pieces per slice.
"""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

from cudanextgenpb_amd import native

from test_zz_no_alloc import hip, solve_noalloc

pytestmark = pytest.mark.gpu


def system(n, form, rng):
    if form == "part":  # a grid, with rows in no pattern at its start
        m = n // 8
        i = np.concatenate([np.arange(n - d) for d in (1, 70, 4900)] + [rng.integers(0, m, 8 * m)])
        j = np.concatenate([np.arange(d, n) for d in (1, 70, 4900)] + [rng.integers(0, m, 8 * m)])
        v = -rng.uniform(0.5, 1.0, len(i))
    elif form == "random":  # about 17 entries a row, in no pattern
        i, j = rng.integers(0, n, 8 * n), rng.integers(0, n, 8 * n)
        v = -rng.uniform(0.5, 1.0, 8 * n)
    else:
        offs = {"constant": (1, 9, 81), "vary": (1, 9, 81), "full": (1, 2, 3, 5, 7, 9), "over": range(1, 8)}[form]
        i = np.concatenate([np.arange(max(0, n - d)) for d in offs])
        j = i + np.concatenate([np.full(max(0, n - d), d) for d in offs])
        v = -np.ones(len(i)) if form == "constant" else -rng.uniform(0.5, 1.0, len(i))
        if form == "constant":  # lines of 9 rows: no coupling across their ends
            v[(j - i == 1) & (i % 9 == 8)] = 0.0
    keep = (i != j) & (v != 0)
    A = sp.coo_matrix((v[keep], (i[keep], j[keep])), shape=(n, n)).tocsr()
    A = A + A.T
    d = 2.0 * max(abs(A).sum(axis=1).max(), 1.0) + np.zeros(n)
    if form == "vary":
        d *= rng.uniform(0.99, 1.01, n)
    A = (A + sp.diags(d)).tocsr()
    A.sum_duplicates()
    A.sort_indices()
    return A


@pytest.mark.parametrize("n,form", [(n, f) for n in (1, 63, 64, 65, 255, 257, 1000, 1025, 2049, 4096, 4097, 70001)
                                    for f in ("constant", "vary", "full", "over", "random")] +
                         [(n, "part") for n in (262145, 300000, 340000, 524288, 700001)])
def test_forms(n, form):
    rng = np.random.default_rng(n)
    A = system(n, form, rng)
    b = rng.standard_normal(n)
    S = SimpleNamespace(n=n, rowptr=A.indptr, col=A.indices, val=A.data, rhs=b)
    rc, x, st = solve_noalloc(hip(), S, 1e-13)
    assert rc == 0 and st["status"] == 0
    ref = spl.spsolve(A.tocsc(), b) if form not in ("random", "part") else None
    if ref is not None:
        assert np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref)
    assert np.linalg.norm(A @ x - b) <= 1e-12 * np.linalg.norm(b)


def test_more_iterations_than_one_launch():
    """A chain whose CG needs more iterations than one launch of the small-system kernel
    takes."""
    n = 4000
    A = sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1]).tocsr()
    b = np.zeros(n)
    b[n // 3] = 1.0
    S = SimpleNamespace(n=n, rowptr=A.indptr, col=A.indices, val=A.data, rhs=b)
    rc, x, st = solve_noalloc(hip(), S, 1e-13)
    # a source at row k: the solution is exact once the residual has run through the chain
    assert rc == 0 and 1024 < st["iterations"] <= 2 * n
    i = np.arange(1, n + 1)
    s = n // 3 + 1
    ref = np.where(i <= s, i * (n + 1 - s), s * (n + 1 - i)) / (n + 1)
    # condition number about 4 (n + 1)^2 / pi^2 = 6.5e6
    assert np.linalg.norm(x - ref) <= 6.5e6 * 1e-13 * np.linalg.norm(ref)


@pytest.mark.parametrize("n,form", [(1000, "vary"), (4096, "full"), (4096, "over"), (4097, "vary")])
def test_profiling_changes_no_result(n, form):
    """Solves in one block and solves of three launches per iteration, with products timed
    and without."""
    rng = np.random.default_rng(n)
    A = system(n, form, rng)
    with native.Context(0) as c:
        c.set_csr(A.indptr, A.indices, A.data, rng.standard_normal(n))
        ref, st = c.solve(native.PREC_FP64, tol=1e-13)
        c.set_profiling(True)
        got, sp_ = c.solve(native.PREC_FP64, tol=1e-13)
        k = c.kernel_stats(native.PREC_FP64)
        c.set_profiling(False)
        again, _ = c.solve(native.PREC_FP64, tol=1e-13)
    assert np.array_equal(got, ref) and np.array_equal(again, ref)
    assert {**sp_, "ms_solve": 0} == {**st, "ms_solve": 0}
    assert k["launches"] == (st["iterations"] + 3) // 8 and k["total_ms"] > 0.0
