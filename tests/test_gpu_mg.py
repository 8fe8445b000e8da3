"""The multigrid preconditioner of the mixed solve (csrc/ngpb_mg.hip).

Each system's mixed potential (true residual 1e-10 of ||b||) against its FP64 solve to
1e-12: the difference is bounded by the condition of the scaled operator times 1e-10;
1e-8 leaves a factor of 300 over the largest measured (3e-11 on meshes of this size).
Sizes where a level can go wrong: 3 cells an axis (one coarse
interior node), odd counts (the last coarse cell reaches past the box), boxes of uneven
sides (a last level of several nodes), four refinement levels (nodes that live on levels
2 to 4), rows in bands. Where the preconditioner does not apply (a lattice too sparse, a
Dirichlet set other than the box faces, an operator loaded as CSR, no memory for it) it is
not in use, nothing is held for it, and the Jacobi-scaled iteration gives the potential.
"""
import dataclasses

import numpy as np
import pytest

from cudanextgenpb_amd import native, workload as W
from cudanextgenpb_amd.batch import prepare

pytestmark = pytest.mark.gpu


def box_spec(n, h=0.5, levels=0, bands=(), atoms=3):
    n = np.asarray(n, np.int64)
    half = 0.5 * n * h
    rng = np.random.default_rng(int(n.sum()))
    xyz = rng.uniform(-0.4, 0.4, (atoms, 3)) * half
    a = W.Atoms(xyz, rng.uniform(0.3, 0.45, atoms) * half.min(), rng.normal(0.0, 0.5, atoms))
    return W.Spec("box", W.Physics(), a, -half, h, n, levels, tuple(bands), 2, W.P4EST_TOL * n[0] * h)


def solve_both(ctx, multigrid=True):
    phi64, st64 = ctx.solve(native.PREC_FP64, tol=1e-12)
    phi, st = ctx.solve(native.PREC_MIXED, tol=1e-10)
    rel = np.linalg.norm(phi - phi64) / np.linalg.norm(phi64)
    print(f"   n={ctx.n}: FP64 {st64['iterations']} it, mixed {st['iterations']} it, phi rel {rel:.1e}", flush=True)
    assert st["status"] == 0 and st["relres"] <= 1e-10 and rel <= 1e-8
    info = ctx.multigrid_info()
    assert info["in_use"] == multigrid and (info["bytes"] > 0) == multigrid
    return phi, st


@pytest.mark.parametrize("n", [(3, 3, 3), (4, 4, 4), (5, 4, 7), (9, 8, 11), (17, 33, 16), (12, 40, 96), (64, 64, 64),
                               (61, 61, 61)])
def test_uniform_boxes(n):
    print(f"[mg] uniform box {n}", flush=True)
    p = prepare(box_spec(n))
    phi, st = solve_both(p.ctx)
    assert st["iterations"] <= 60
    again, _ = p.ctx.solve(native.PREC_MIXED, tol=1e-10)
    assert np.array_equal(phi, again)
    p.ctx.close()


@pytest.mark.parametrize("levels,bands,n", [(1, (1.0,), 40), (2, (1.0, 2.5), 48), (3, (1.0, 2.5, 5.0), 64),
                                            (4, (1.0, 2.0, 4.0, 8.0), 64)])
def test_octree_levels(levels, bands, n):
    print(f"[mg] {levels} refinement levels", flush=True)
    p = prepare(box_spec((n, n, n), levels=levels, bands=bands, atoms=4))
    phi, st = solve_both(p.ctx)
    assert st["iterations"] <= 60
    p.ctx.set_row_order(4)
    banded, _ = p.ctx.solve(native.PREC_MIXED, tol=1e-10)
    assert np.linalg.norm(banded - phi) <= 1e-8 * np.linalg.norm(phi)
    p.ctx.close()


def test_sparse_lattice_uses_jacobi():
    """More than 32 finest-lattice vertices per node: the dense transfer array is not built."""
    p = prepare(box_spec((192, 192, 192), h=0.25, levels=4, bands=(0.1, 0.1, 0.1, 0.1), atoms=1))
    assert 193 ** 3 > 32 * p.n
    solve_both(p.ctx, multigrid=False)
    p.ctx.close()


def test_other_dirichlet_sets_and_csr_use_jacobi():
    P = W.three_spheres()
    ctx = native.Context(0)
    ctx.set_physics(P.physics)
    ctx.set_mesh(P.mesh)
    ctx.set_rays(P.rays)
    ctx.create_markers()
    ctx.set_charges(P.atoms.xyz, P.atoms.q, P.owner)
    inner = int(np.argmin(np.abs(P.mesh.node_xyz).sum(axis=1)))
    nodes = np.append(P.mesh.bnd_nodes, inner).astype(np.int32)  # one fixed node inside
    ctx.set_dirichlet(nodes, np.linspace(0.0, 0.1, len(nodes)))
    ctx.assemble()
    solve_both(ctx, multigrid=False)
    csr = ctx.export_csr()
    ctx.close()
    other = native.Context(0)
    other.set_csr(*csr)
    solve_both(other, multigrid=False)
    other.close()


def test_no_memory_uses_jacobi():
    """A bound on its memory that any of its allocations can run into: the solve goes on
    as with Jacobi scaling from the start, alone and in a batch."""
    p = prepare(box_spec((48, 48, 48), levels=2, bands=(1.0, 2.5)))
    _, st = solve_both(p.ctx)
    full = p.ctx.multigrid_info()["bytes"]
    p.ctx.set_multigrid(cycle_iters=0)
    phi, stj = solve_both(p.ctx, multigrid=False)
    assert stj["iterations"] > 2 * st["iterations"]
    n = p.n
    for bound in (1, full // 2, full - 12 * n - 1, full - 8 * n, full - 1):
        print(f"[mg] {bound} of {full} bytes", flush=True)
        p.ctx.set_multigrid(max_bytes=bound)
        got, s = solve_both(p.ctx, multigrid=False)
        assert np.array_equal(got, phi) and s["iterations"] == stj["iterations"]
        with native.Batch(0, max_systems=1, tol=1e-10) as b:
            slot = b.add(p.ctx)
            b.run(1000)
            done, sb = b.status(slot)
            b.remove(slot)
        assert done and sb["status"] == 0 and not p.ctx.multigrid_info()["in_use"]
        assert np.linalg.norm(p.ctx.get_phi() - phi) <= 1e-8 * np.linalg.norm(phi)
    p.ctx.set_multigrid(max_bytes=full)
    solve_both(p.ctx)
    p.ctx.close()


def test_host_mesh_equals_device_mesh():
    """The hierarchy is found from the mesh arrays alone: a mesh handed over by the caller
    and the same mesh built on the device give the same potential bit for bit."""
    P = W.three_spheres()
    out = []
    for device_mesh in (False, True):
        p = prepare(P, device_mesh=device_mesh)
        out.append(p.ctx.solve(native.PREC_MIXED, tol=1e-10))
        p.ctx.close()
    assert out[0][1]["iterations"] == out[1][1]["iterations"] <= 60
    assert np.array_equal(out[0][0], out[1][0])


def solve_batch(ctxs, maxiter=100000, inner=8):
    """Potentials and statistics of the contexts solved in one batch, and its replays."""
    with native.Batch(0, max_systems=len(ctxs), tol=1e-10, maxiter=maxiter, inner_per_replay=inner) as b:
        slots = [b.add(c) for c in ctxs]
        replays = b.solve_all(5000)
        out = []
        for s, c in zip(slots, ctxs):
            done, st = b.status(s)
            assert done
            b.remove(s)
            out.append((c.get_phi(), st))
    return out, replays


def test_cycle_that_does_not_converge():
    """A limit on the iterations of a cycle ends it early: the solve goes on from its x
    with Jacobi scaling, within the iteration limit of the whole solve, and other systems
    of a batch are not touched by it."""
    p = prepare(box_spec((48, 48, 48), levels=2, bands=(1.0, 2.5)))
    other = prepare(box_spec((17, 33, 16)))
    phi64, _ = p.ctx.solve(native.PREC_FP64, tol=1e-12)

    def close(phi):
        return np.linalg.norm(phi - phi64) <= 1e-8 * np.linalg.norm(phi64)

    p.ctx.set_multigrid(cycle_iters=0)
    _, jac = p.ctx.solve(native.PREC_MIXED, tol=1e-10)
    [(_, jac_b)], _ = solve_batch([p.ctx])
    [(ref_other, _)], _ = solve_batch([other.ctx])
    for limit in (1, 3, 5):
        p.ctx.set_multigrid(cycle_iters=limit)
        phi, st = p.ctx.solve(native.PREC_MIXED, tol=1e-10)
        [(alone, sa)], _ = solve_batch([p.ctx])
        [(mix, sm), (phi_other, _)], _ = solve_batch([p.ctx, other.ctx])
        print(f"[mg] cycles of {limit}: {st['iterations']} it, batch {sa['iterations']} it "
              f"(Jacobi {jac['iterations']} and {jac_b['iterations']})", flush=True)
        assert p.ctx.multigrid_info()["in_use"]
        for f, s in ((phi, st), (alone, sa), (mix, sm)):
            assert s["status"] == 0 and s["relres"] <= 1e-10 and close(f)
        assert np.array_equal(alone, mix) and sa["iterations"] == sm["iterations"]
        assert np.array_equal(phi_other, ref_other)
        if limit > 1:  # what the first cycle gained is kept
            assert limit < st["iterations"] < jac["iterations"] + limit
            assert limit < sa["iterations"] < jac_b["iterations"] + limit
        # the iterations of the ended cycle count towards the limit
        _, s20 = p.ctx.solve(native.PREC_MIXED, tol=1e-10, maxiter=20, raise_on_noconv=False)
        [(_, b20)], replays = solve_batch([p.ctx], maxiter=20, inner=1)
        for s in (s20, b20):
            assert s["status"] == 4 and s["iterations"] == 20
        assert replays <= 20 + b20["replacements"] + 2
    p.ctx.close()
    other.ctx.close()


def test_batch_reports_the_iteration_it_runs():
    p = prepare(box_spec((17, 33, 16)))
    seen = []
    for cycles in (100, 0):
        p.ctx.set_multigrid(cycle_iters=cycles)
        _, st = p.ctx.solve(native.PREC_MIXED, tol=1e-10)
        [(_, sb)], _ = solve_batch([p.ctx])
        assert sb["bytes_per_iter"] == st["bytes_per_iter"]
        seen.append(st["bytes_per_iter"])
    assert seen[0] > 2 * seen[1]  # three products and the levels against one product
    p.ctx.close()
