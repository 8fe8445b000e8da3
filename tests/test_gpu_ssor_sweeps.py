"""SSOR sweeps on sparsity patterns that reach every path of the level-ordered sweeps
(csrc/ngpb_lis.hip), bit-identical to the oracle's sequential sweeps:

* triangles without entries, from one row up, and one level of all rows (wider than a
  one-block run): launched on their own;
* one row per level (a chain; neighbours in the LDS window only);
* chains with links far behind (neighbours older than the 8192-position window, read
  from memory) and to the first rows, links at the window's edge, and levels of one full
  piece (512 rows) linked 15, 16 and 17 levels back;
* few and many levels that are all launched;
* rows with more neighbours than are read together (4, 8, 16), and random patterns whose
  levels are narrow at the ends and wide in the middle (runs between launches);
* levels of 255 .. 2049 rows around the piece size (512 rows) and the widths from which
  levels are launched one by one;
* levels that are launched between runs for their length or for a row too long for a
  piece (2048 entries).
"""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle as O
from cudanextgenpb_amd import native

pytestmark = pytest.mark.gpu


def system(n, pairs, seed):
    """Symmetric, diagonally dominant CSR with the given off-diagonal pairs (i > j)."""
    rng = np.random.default_rng(seed)
    pairs = np.unique(np.asarray(pairs, np.int64).reshape(-1, 2), axis=0)
    v = -rng.uniform(0.1, 1.0, len(pairs))
    A = sp.coo_matrix((v, (pairs[:, 0], pairs[:, 1])), shape=(n, n)).tocsr()
    A = A + A.T
    A = (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + rng.uniform(0.5, 1.5, n))).tocsr()
    A.sort_indices()
    return O.System(n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.copy(), np.ones(n))


def layered(width, layers, links, seed, far=0):
    """Layers of `width` rows, each row linked to `links` rows of the layer before and,
    for `far` of the rows, to one row of any earlier layer."""
    rng = np.random.default_rng(seed)
    out = []
    for l in range(1, layers):
        i = np.arange(l * width, (l + 1) * width)
        for _ in range(links):
            out.append(np.stack([i, rng.integers((l - 1) * width, l * width, width)], 1))
        if far:
            k = rng.choice(i, size=min(far, width), replace=False)
            out.append(np.stack([k, rng.integers(0, l * width, len(k))], 1))
    return system(width * layers, np.concatenate(out), seed)


def cases():
    for n in (1, 2, 64, 513, 2048, 2049, 5000):
        yield f"diagonal_{n}", system(n, np.zeros((0, 2)), 1)
    yield "chain", system(3000, [(i, i - 1) for i in range(1, 3000)], 2)
    n = 30000
    far = [(i, i - 1) for i in range(1, n)] + [(i, i - 20000) for i in range(20000, n, 7)] + [(i, 0) for i in range(2, n, 11)]
    yield "far_chain", system(n, far, 3)
    n = 9000
    edge = [(i, i - 1) for i in range(1, n)] + [(i, i - d) for d in (8190, 8191, 8192, 8193) for i in range(d, n, 3)]
    yield "window_edge", system(n, edge, 6)
    i = np.arange(512, 512 * 40)
    back = [np.stack([i, i - 512], 1)] + [np.stack([i, i - 512 * k], 1)[i >= 512 * k] for k in (15, 16, 17)]
    yield "full_pieces", system(512 * 40, np.concatenate(back), 7)
    yield "long_rows", layered(100, 30, 13, 4)
    for width in (255, 256, 257, 512, 513, 1024, 1025, 2048, 2049):
        yield f"layers_{width}", layered(width, 12, 3, width, far=40)
    for levels in (2, 3, 8, 9):
        yield f"wide_levels_{levels}", layered(6000, levels, 4, levels, far=100)
    rng = np.random.default_rng(9)
    # narrow levels of short rows, then wide levels of long ones, twice over
    S, base = [], 0
    for width, layers, links in ((40, 30, 2), (1500, 6, 12), (40, 30, 2), (1500, 6, 12), (40, 5, 2)):
        for l in range(layers):
            i = np.arange(base, base + width)
            if base:
                S += [np.stack([i, rng.integers(max(0, base - 40), base, width)], 1) for _ in range(links)]
            base += width
    yield "mixed_levels", system(base, np.concatenate(S), 8)
    n = 6000  # one row coupled to 3,000 before it
    long_row = [(i, i - 1) for i in range(1, n)] + [(5000, i) for i in range(0, 4999, 1) if i % 5 < 3]
    yield "row_over_a_piece", system(n, long_row, 10)
    i = rng.integers(1, 60000, 200000)
    yield "random", system(60000, np.stack([i, (i * rng.random(len(i))).astype(np.int64)], 1), 5)


@pytest.mark.parametrize("name,S", list(cases()), ids=lambda v: v if isinstance(v, str) else "")
def test_sweeps_bit_identical(name, S):
    r = np.random.default_rng(7).standard_normal(S.n)
    ctx = native.Context(0)
    ctx.set_csr(S.rowptr, S.col, S.val, S.rhs)
    for w in (0.51, 1.3):
        print(f"[ssor sweep] {name} n={S.n} w={w}", flush=True)
        assert np.array_equal(ctx.precond_apply(r, native.PRECON_SSOR, w), O.ssor_apply(S, w, r))
    ctx.close()
