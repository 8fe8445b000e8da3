"""Device blocks of destroyed contexts are reused by later ones (the pool behind the
device buffers):

* contexts made, used and destroyed from several threads at once, with sizes that
  alternate, give the potentials and energies of contexts that took fresh memory, bit for
  bit (reused blocks hold old data, so a buffer read before it is written would show);
* the memory a process holds after many contexts is bounded by what its first ones needed;
* trim_pool gives the idle blocks back to the driver, in part and in whole.
"""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from cudanextgenpb_amd import native, workload as W
from cudanextgenpb_amd.batch import prepare

from test_gpu_block_cache import _free_bytes, _hip, _spec

pytestmark = pytest.mark.gpu


def _solve(spec, precision, probe):
    p = prepare(spec, probe=probe)
    phi, _ = p.ctx.solve(precision, tol=1e-10)
    out = phi, p.ctx.energy()["polar"], p.ctx.phi_on_atoms(p.atoms)
    p.ctx.close()
    return out


def test_reused_blocks_across_threads():
    jobs = [(_spec(i % 3), pr, probe) for i in range(3) for pr in (native.PREC_MIXED, native.PREC_FP64)
            for probe in (0.0, 1.4)]
    ref = [_solve(*j) for j in jobs]
    with ThreadPoolExecutor(4) as ex:
        for r in range(3):
            print(f"[block pool] round {r}", flush=True)
            order = np.random.default_rng(r).permutation(len(jobs))
            for k, got in zip(order, ex.map(lambda k: _solve(*jobs[k]), order)):
                for name, a, b in zip(("potential", "energy", "at atoms"), got, ref[k]):
                    d = np.abs(np.asarray(a) - np.asarray(b))
                    assert np.array_equal(a, b), (jobs[k][0].name, "mixed" if jobs[k][1] else "fp64", jobs[k][2], name,
                                                  int((d > 0).sum()), float(d.max()))


def test_pool_does_not_grow():
    hip = _hip()
    for S in (_spec(0), _spec(2)):
        _solve(S, native.PREC_MIXED, 1.4)
    free0 = _free_bytes(hip)
    for _ in range(5):
        for S in (_spec(0), _spec(2)):
            _solve(S, native.PREC_MIXED, 1.4)
    assert free0 - _free_bytes(hip) < 64 * 2**20


def test_pool_is_given_back():
    hip = _hip()
    big = _spec(2)
    ref = _solve(big, native.PREC_MIXED, 1.4)
    held = native.trim_pool(0, 1 << 60)
    free0 = _free_bytes(hip)
    assert held > 32 * 2**20
    half = native.trim_pool(0, held // 2)
    assert 0 < half <= held // 2
    assert native.trim_pool(0, 1 << 60) == half
    got = _solve(big, native.PREC_MIXED, 1.4)  # part of its blocks from the pool, part new
    assert all(np.array_equal(a, b) for a, b in zip(got, ref))
    assert native.trim_pool(0) == 0
    # the driver rounds blocks; most of what was held must be free again
    assert _free_bytes(hip) - free0 > held // 2
    got = _solve(big, native.PREC_MIXED, 1.4)
    assert all(np.array_equal(a, b) for a, b in zip(got, ref))
