"""The work that programs built on this library spend their time on, as measurable cases.

A case is a dict of plain values. Its "kind" names the call sequence:

  csr      ngpb_solve_csr_noalloc on a device CSR the caller holds (code that cannot
           allocate): the smallest calls, where launches and polls count
  request  one molecule from its atoms to potential and energies on a fresh context:
           octree, rays, markers, owners, charges, boundary values, assembly, solve,
           energy, potential at the atoms (what the serving loop does per request)
  step     a new charge set on a resident mesh (titration and pKa scans): markers,
           charges, numeric assembly, solve, energy
  driver   the reference driver's flow: mesh, rays and owners handed over as arrays,
           its member functions in order, with a LIS option string
  batch    many ligands assembled beforehand, solved together with their energies
  outputs  energies, potentials and fields at the atoms for a potential in hand

Molecules come from the synthetic generators of the configurations (globular packing of
2 A minimum separation, the large complex without one, ligands on uniform grids). The
case fixes the reference conformation and its mesh; the seed displaces every atom (a
snapshot of a trajectory on the common grid) and draws the charges, so two seeds share
sizes and nothing else.
"""
import ctypes
import dataclasses
import math

import numpy as np
import torch

from cudanextgenpb_amd import native, workload as W
from cudanextgenpb_amd.batch import BatchedSolver, prepare_many
from cudanextgenpb_amd.pb import PoissonBoltzmann

LIS_DEFAULT = "-p ssor -ssor_omega 0.51 -i cgs -tol 1.e-6"  # the reference's default options
LIS_JACOBI = "-i cg -p jacobi -tol 1.e-10 -maxiter 100000"
LIGAND_H = 0.4


def listed():
    return [
        # 16^3 interior nodes around one ion: a solve of a few thousand rows between other GPU work
        {"name": "csr_16", "kind": "csr", "m": 16},
        # 100^3: close to the largest system that entry point takes (2^20 rows)
        {"name": "csr_100", "kind": "csr", "m": 100},
        # one ligand of the batched configuration on its uniform 0.4 A grid, served alone
        {"name": "request_ligand", "kind": "request", "atoms": 45, "grid": 64, "molecule": 7, "precision": "mixed"},
        # the smallest request of the serving stream: 50 atoms, 0.5 A leaves within 3 A
        {"name": "request_50", "kind": "request", "atoms": 50, "grid": 0, "fine": 3.0, "mid": 6.0, "molecule": 11,
         "precision": "mixed"},
        # the headline molecule: 2,500 atoms, 8.0M unknowns, solvent-excluded surface
        {"name": "request_2500", "kind": "request", "atoms": 2500, "grid": 0, "fine": 39.0, "mid": 45.0,
         "molecule": 20502, "precision": "mixed"},
        # the headline step: resident 8.0M-unknown mesh, mixed precision
        {"name": "step_2500", "kind": "step", "atoms": 2500, "grid": 0, "fine": 39.0, "mid": 45.0,
         "molecule": 20502, "precision": "mixed"},
        # the largest configuration: 40,000 atoms, 63M unknowns
        {"name": "step_40000", "kind": "step", "atoms": 40000, "grid": 0, "fine": 58.0, "mid": 64.0,
         "molecule": 40003, "precision": "mixed"},
        # an ion on a uniform 129^3 grid (0.25 A) in FP64, the plain drop-in for -i cg -p jacobi
        {"name": "step_ion_fp64", "kind": "step", "atoms": 1, "grid": 128, "molecule": 0, "precision": "fp64"},
        # the reference's default options on a protein of 600 atoms, every array handed over by the driver
        {"name": "driver_ssor", "kind": "driver", "atoms": 600, "fine": 3.0, "mid": 6.0, "molecule": 31,
         "options": LIS_DEFAULT},
        # the FP64 Jacobi-CG option string on a larger protein
        {"name": "driver_jacobi", "kind": "driver", "atoms": 4000, "fine": 3.0, "mid": 6.0, "molecule": 32,
         "options": LIS_JACOBI},
        # the 128 ligands of the default benchmark line
        {"name": "batch_128", "kind": "batch", "systems": 128, "first": 0},
        # phi_on_atoms.txt, pot_field.dat and the energies of a 2,500-atom protein
        {"name": "outputs_2500", "kind": "outputs", "atoms": 2500, "fine": 3.0, "mid": 6.0, "molecule": 41},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["csr", "request", "request", "ligand", "step", "driver", "batch", "outputs"])
    mol = rng.randrange(100, 1 << 20)
    bands = rng.choice([(3.0, 6.0), (2.0, 5.0), (6.0, 9.0)])
    if kind == "csr":
        return {"kind": "csr", "m": _log(rng, 12, 101)}
    if kind == "ligand":
        return {"kind": "request", "atoms": rng.randrange(20, 81), "grid": rng.randrange(48, 97), "molecule": mol,
                "precision": rng.choice(["mixed", "fp64"])}
    if kind == "request":
        return {"kind": "request", "atoms": _log(rng, 50, 20000), "grid": 0, "fine": bands[0], "mid": bands[1],
                "molecule": mol, "precision": rng.choice(["mixed", "mixed", "fp64"])}
    if kind == "step":
        if rng.random() < 0.3:
            return {"kind": "step", "atoms": 1, "grid": rng.randrange(60, 161), "molecule": 0,
                    "precision": rng.choice(["mixed", "fp64"])}
        return {"kind": "step", "atoms": _log(rng, 200, 5000), "grid": 0, "fine": rng.uniform(3.0, 20.0), "mid": 26.0,
                "molecule": mol, "precision": "mixed"}
    if kind == "driver":
        ssor = rng.random() < 0.5
        return {"kind": "driver", "atoms": _log(rng, 50, 800 if ssor else 6000), "fine": bands[0], "mid": bands[1],
                "molecule": mol, "options": LIS_DEFAULT if ssor else LIS_JACOBI}
    if kind == "batch":
        return {"kind": "batch", "systems": _log(rng, 2, 96), "first": rng.randrange(0, 400)}
    return {"kind": "outputs", "atoms": _log(rng, 50, 6000), "fine": bands[0], "mid": bands[1], "molecule": mol}


# ------------------------------------------------------------------ molecules
def _reference(case):
    """The case's reference conformation with the mesh parameters made from it (a Spec)."""
    n = case["atoms"]
    if case.get("grid"):  # uniform grid: ligand (0.4 A, extent box / 1.6) or ion (0.25 A)
        h, m = (0.25, case["grid"]) if n == 1 else (LIGAND_H, case["grid"])
        if n == 1:
            atoms = W.Atoms(np.zeros((1, 3)), np.array([2.0]), np.array([1.0]))
        else:
            ball = 0.5 * m * h / 1.6 - 1.9
            atoms = W.make_atoms(case["molecule"], n, [0.0] * 3, [ball] * 3, 1.2, 1.2, 1.9, 0.3, float("nan"))
        return W.Spec("uniform", W.Physics(), atoms, np.full(3, -0.5 * m * h), h, np.full(3, m, np.int64), 0, (), 2,
                      W.P4EST_TOL * m * h)
    if n >= 40000:
        return W.large_spec(n_atoms=n, fine_band=case["fine"], mid_band=case["mid"])
    return W.globular_spec(seed=case["molecule"], n_atoms=n, ball_radius=20.0 * (n / 2500.0) ** (1 / 3),
                           fine_band=case["fine"], mid_band=case["mid"], qnet=round(-3.0 * n / 2500.0))


def _snapshot(spec, seed):
    """Displaced atoms (0.1 A per coordinate, at most 0.3 A) with newly drawn charges."""
    rng = np.random.Generator(np.random.PCG64(seed))
    a = spec.atoms
    xyz = a.xyz + np.clip(rng.normal(0.0, 0.1, a.xyz.shape), -0.3, 0.3)
    q = rng.normal(0.0, 0.35, a.n)
    q = np.array([rng.uniform(0.5, 1.5)]) if a.n == 1 else q + (float(round(a.q.sum())) - q.sum()) / a.n
    return W.Atoms(np.ascontiguousarray(xyz), a.r.copy(), q)


def _probe(case):
    return 0.0 if case.get("grid") else 1.4  # uniform configurations use the sphere union


def _precision(case):
    return native.PREC_MIXED if case["precision"] == "mixed" else native.PREC_FP64


def _unknowns(case):
    """Estimated unknowns of the case's mesh: balls of the finest and the next leaves."""
    if case["kind"] == "csr":
        return case["m"] ** 3
    if case["kind"] == "batch":
        return 400_000 * case["systems"]
    if case.get("grid"):
        return (case["grid"] + 1) ** 3
    h = 0.35 if case["atoms"] >= 40000 else 0.5
    r = 27.0 if case["atoms"] >= 40000 else 20.0 * (case["atoms"] / 2500.0) ** (1 / 3)
    half = 3.0 * (r + 2.0)
    fine = min(4.19 * (r + 2.0 + case["fine"]) ** 3, (2 * half) ** 3)
    mid = min(4.19 * (r + 2.0 + case["mid"]) ** 3, (2 * half) ** 3) - fine
    return int(fine / h**3 + mid / (2 * h) ** 3 + ((2 * half) ** 3 - fine - mid) / (4 * h) ** 3)


# ------------------------------------------------------------------ csr systems
def _blob(m, seed, device):
    """Face conductances of a two-dielectric grid of (m + 2)^3 nodes at 0.4 A (a random
    union of balls, permittivity 2 in 80), and charges on interior nodes."""
    g = torch.Generator().manual_seed(int(seed))
    n = m + 2
    c = (torch.rand(20, 3, generator=g, dtype=torch.float64) * 0.5 + 0.25).mul(n - 1).to(device)
    r = (torch.rand(20, generator=g, dtype=torch.float64) * 0.06 + 0.05).mul(n).to(device)
    ax = torch.arange(n, dtype=torch.float64, device=device)
    inside = torch.zeros(n, n, n, dtype=torch.bool, device=device)
    for k in range(20):
        d = [(ax - c[k, i]) ** 2 for i in range(3)]
        inside |= d[2][:, None, None] + d[1][None, :, None] + d[0][None, None, :] < r[k] ** 2
    eps = torch.full((n, n, n), 80.0, dtype=torch.float64, device=device).masked_fill_(inside, 2.0)
    mean = lambda a, b: 2.0 / (1.0 / a + 1.0 / b)
    cz, cy, cx = mean(eps[1:], eps[:-1]), mean(eps[:, 1:], eps[:, :-1]), mean(eps[:, :, 1:], eps[:, :, :-1])
    mass = (~inside).double()[1:-1, 1:-1, 1:-1] * (80.0 * 0.0157 * 0.16)
    rhs = torch.zeros(m, m, m, dtype=torch.float64)
    at = torch.randint(0, m, (60, 3), generator=g)
    rhs.index_put_((at[:, 0], at[:, 1], at[:, 2]), torch.randn(60, generator=g, dtype=torch.float64) * 50.0,
                   accumulate=True)
    i = slice(1, -1)
    # conductance to the lower and the upper neighbour of every interior node, per axis
    lo = [cz[:-1, i, i], cy[i, :-1, i], cx[i, i, :-1]]
    hi = [cz[1:, i, i], cy[i, 1:, i], cx[i, i, 1:]]
    return lo, hi, sum(lo) + sum(hi) + mass, rhs.to(device)


def _csr(m, seed, device):
    lo, hi, diag, rhs = _blob(m, seed, device)
    n = m**3
    row = torch.arange(n, device=device).view(m, m, m)
    z, y, x = torch.meshgrid(*[torch.arange(m, device=device)] * 3, indexing="ij")
    pos, step = [z, y, x], [m * m, m, 1]
    cols, vals, keep = [], [], []
    for a in range(3):  # ascending columns: -z -y -x diagonal +x +y +z
        cols.append(row - step[a])
        vals.append(-lo[a])
        keep.append(pos[a] > 0)
    cols.append(row)
    vals.append(diag)
    keep.append(torch.ones_like(row, dtype=torch.bool))
    for a in (2, 1, 0):
        cols.append(row + step[a])
        vals.append(-hi[a])
        keep.append(pos[a] < m - 1)
    cols, vals, keep = (torch.stack([t.reshape(n) for t in v], 1) for v in (cols, vals, keep))
    ptr = torch.zeros(n + 1, dtype=torch.int32, device=device)
    ptr[1:] = torch.cumsum(keep.sum(1), 0)
    return ptr, cols[keep].int().contiguous(), vals[keep].contiguous(), rhs.reshape(n).contiguous()


# ------------------------------------------------------------------ prepare / run
def _inputs(ctx, spec, atoms, probe):
    """A molecule from its atoms to boundary values on the device; the mesh is the
    reference conformation's."""
    ctx.set_physics(spec.physics)
    ctx.build_octree(*spec.generator_params(), spec.atoms.xyz, spec.atoms.r)
    if probe > 0.0:
        ctx.cast_rays_ses(atoms.xyz, atoms.r, probe)
    else:
        ctx.cast_rays(atoms.xyz, atoms.r)
    ctx.create_markers()
    ctx.set_charges(atoms.xyz, atoms.q, ctx.locate_atoms(atoms.xyz, spec.atom_tol))
    ctx.dirichlet_values(spec.bc_type)


def _batch_specs(case, seed):
    out = []
    for k in range(case["systems"]):
        spec = W.ligand_spec(case["first"] + k)
        out.append(dataclasses.replace(spec, atoms=_snapshot(spec, seed * 1000 + k)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "csr":
        ptr, col, val, rhs = _csr(case["m"], seed, "cuda")
        opts = native.SolveOpts(native.PREC_FP64, 1e-10, 100000, 1e-3, 32, native.SOLVER_CG, native.PRECON_JACOBI, 1.0)
        return {"kind": kind, "ptr": ptr, "col": col, "val": val, "rhs": rhs, "x": torch.empty_like(rhs), "opts": opts}
    if kind == "batch":
        preps = prepare_many(_batch_specs(case, seed))
        bs = BatchedSolver(0, max_systems=len(preps), tol=1e-10)
        for p in preps:
            bs.add(p)
        bs.autotune()
        for slot in list(bs.slots):
            bs.batch.remove(slot)
            del bs.slots[slot]
        return {"kind": kind, "preps": preps, "solver": bs}
    if kind == "driver":
        P = W.globular(seed=case["molecule"], n_atoms=case["atoms"],
                       ball_radius=20.0 * (case["atoms"] / 2500.0) ** (1 / 3), fine_band=case["fine"],
                       mid_band=case["mid"], qnet=round(-3.0 * case["atoms"] / 2500.0))
        atoms = _snapshot(P, seed)
        P = dataclasses.replace(P, atoms=atoms, rays=W.cast_rays(P.mesh, atoms),
                                owner=W.locate_atoms(P.mesh, atoms, P.atom_tol))
        return {"kind": kind, "problem": P, "options": case["options"]}
    spec = _reference(case)
    atoms = _snapshot(spec, seed)
    state = {"kind": kind, "spec": spec, "atoms": atoms, "probe": _probe(case)}
    if kind == "request":
        return dict(state, precision=_precision(case))
    ctx = native.Context(0)
    _inputs(ctx, spec, atoms, state["probe"])
    ctx.assemble()
    state["ctx"] = ctx
    if kind == "step":
        return dict(state, precision=_precision(case))
    # outputs: a screened Coulomb potential on the nodes, as a solver would have left it
    # (the context is given its solution vector by a solve of one iteration)
    ctx.solve(native.PREC_FP64, maxiter=1, want_phi=False, raise_on_noconv=False)
    xyz = torch.from_numpy(ctx.get_mesh()["node_xyz"]).cuda()
    a, q = torch.from_numpy(atoms.xyz).cuda(), torch.from_numpy(atoms.q).cuda()
    eps = native.constants(spec.physics)["eps_out"]
    phi = torch.empty(xyz.shape[0], dtype=torch.float64, device="cuda")
    for k in range(0, xyz.shape[0], 1 << 15):
        d = torch.cdist(xyz[k:k + (1 << 15)], a) + 0.5
        phi[k:k + (1 << 15)] = (torch.exp(-0.125 * d) / d) @ q / eps
    ctx.set_phi(phi.cpu().numpy())
    return state


def _energies(e):
    return {"polar": e["energy_pol"], "ionic": e["energy_react"]}


def run(state):
    kind = state["kind"]
    if kind == "csr":
        s, st = state, native.SolveStats()
        rc = native.lib().ngpb_solve_csr_noalloc(
            0, torch.cuda.current_stream().cuda_stream, s["rhs"].numel(), s["col"].numel(), s["ptr"].data_ptr(),
            s["col"].data_ptr(), s["val"].data_ptr(), s["rhs"].data_ptr(), s["x"].data_ptr(), ctypes.byref(s["opts"]),
            ctypes.byref(st))
        if rc != native.NGPB_OK:
            raise native.NGPBError(rc, "solve_csr_noalloc")
        return s["x"]
    if kind == "request":
        ctx = native.Context(0)
        _inputs(ctx, state["spec"], state["atoms"], state["probe"])
        ctx.assemble()
        phi, _ = ctx.solve(state["precision"], tol=1e-10)
        e = ctx.energy()
        at = ctx.phi_on_atoms(state["atoms"].n)
        ctx.close()
        return {"phi": phi, "at_atoms": at, **_energies(e)}
    if kind == "step":
        ctx, a = state["ctx"], state["atoms"]
        ctx.create_markers()
        ctx.set_charges(a.xyz, a.q, ctx.locate_atoms(a.xyz, state["spec"].atom_tol))
        ctx.assemble()
        phi, _ = ctx.solve(state["precision"], tol=1e-10)
        return {"phi": phi, **_energies(ctx.energy())}
    if kind == "driver":
        pb = PoissonBoltzmann(state["problem"])
        e = pb.run(state["options"])
        phi = pb.phi
        pb.close()
        return {"phi": phi, **_energies(e)}
    if kind == "batch":
        bs = state["solver"]
        for p in state["preps"]:
            bs.add(p)
        res = bs.solve(energies=True)
        phi = np.concatenate([p.ctx.get_phi() for p in state["preps"]])
        e = np.array([[res[p.name]["energy"]["energy_pol"], res[p.name]["energy"]["energy_react"]]
                      for p in state["preps"]])
        return {"phi": phi, "energies": e}
    ctx, n = state["ctx"], state["atoms"].n
    e = ctx.energy()
    table, out = ctx.pot_field(n, 2, 2)
    return {"coulomb": table[:, [0, 3, 4, 5]], "surface": table[:, [1, 2, 6, 7, 8, 9, 10, 11]],
            "at_atoms": ctx.phi_on_atoms(n), **_energies(e), "coulomb_energy": out["coul_energy"]}


def work(case):
    """Inputs read once and outputs written once: the operator and right-hand side where
    the caller holds them, otherwise atoms in and the potential out; one application of
    the operator, and for the atom outputs the source-atom and atom-atom pairs."""
    n = _unknowns(case)
    if case["kind"] == "csr":
        return {"bytes": 7 * 12.0 * n + 20.0 * n, "flops": 14.0 * n}
    if case["kind"] == "outputs":
        sources = 60.0 * case["atoms"] + 2000.0
        return {"bytes": 8.0 * n + 400.0 * sources, "flops": 30.0 * sources * case["atoms"]}
    if case["kind"] in ("step", "batch"):  # the resident matrix pattern and values as well
        return {"bytes": 7 * 12.0 * n + 24.0 * n, "flops": 14.0 * n}
    if case["kind"] == "driver":  # coordinates and leaf corners come from the caller
        return {"bytes": (24.0 + 32.0 + 8.0) * n, "flops": 14.0 * n}
    return {"bytes": 8.0 * n + 40.0 * case["atoms"], "flops": 14.0 * n}


def tolerance(case):
    # Solves stop at a residual of 1e-10 of ||b||; measured against tighter solves, their
    # potentials are up to 1.2e-9 off (100^3 grid; 1.5e-10 on the 63M-unknown mesh) and
    # their energies up to 5e-10. The default LIS options stop at 1e-6: potential 2.6e-6,
    # ionic energy (a small difference) 4e-4 off. The outputs at the atoms are FP64 sums
    # of up to 1e6 terms of both signs.
    if case["kind"] == "outputs":
        return {"rel": 1e-11}
    if case.get("options") == LIS_DEFAULT:
        return {"rel": 1.6e-3}
    return {"rel": 5e-9}


# ------------------------------------------------------------------ 64-bit references
def _cg(lo, hi, diag, rhs, tol=1e-14):
    """Jacobi-CG on the 7-point operator given by its face conductances, in 64 bits."""
    def apply(x):
        y = diag * x
        for a in range(3):
            n = x.shape[a]
            y.narrow(a, 1, n - 1).sub_(lo[a].narrow(a, 1, n - 1) * x.narrow(a, 0, n - 1))
            y.narrow(a, 0, n - 1).sub_(hi[a].narrow(a, 0, n - 1) * x.narrow(a, 1, n - 1))
        return y

    x = torch.zeros_like(rhs)
    for _ in range(3):  # restarts remove the drift of the recursive residual
        r = rhs - apply(x)
        z = r / diag
        p = z.clone()
        rz = (r * z).sum()
        for it in range(20000):
            w = apply(p)
            alpha = rz / (p * w).sum()
            x += alpha * p
            r -= alpha * w
            z = r / diag
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
            if it % 20 == 0 and float(r.norm()) <= tol * float(rhs.norm()):
                break
    return x


def _crossings(lo, hi, xyz, r, axis, t0, t1, upper_inside):
    """Last boundary crossing of the union of balls on each grid edge: lo, hi are the two
    transverse coordinates, [t0, t1] the edge; upper_inside: its upper end is inside."""
    o = [d for d in range(3) if d != axis]
    d2 = (lo[:, None] - xyz[None, :, o[0]]) ** 2 + (hi[:, None] - xyz[None, :, o[1]]) ** 2
    half = (r[None] ** 2 - d2).clamp_min(0).sqrt()
    hit = d2 < r[None] ** 2
    s = torch.where(hit, xyz[None, :, axis] - half, torch.inf)
    e = torch.where(hit, xyz[None, :, axis] + half, -torch.inf)
    out = torch.where((e >= t0[:, None]) & (e <= t1[:, None]), e, -torch.inf).amax(1)  # upper end outside
    start = torch.where((s <= t1[:, None]) & (e > t1[:, None]), s, torch.inf).amin(1)
    for _ in range(20):  # the start of the merged interval that holds the upper end
        start = torch.minimum(start, torch.where(e >= start[:, None], torch.where(s <= start[:, None], s, torch.inf),
                                                 torch.inf).amin(1))
    return torch.where(upper_inside, start, out)


def _uniform(spec, atoms, device):
    """Potential of a sphere-union molecule on a uniform grid (nodes x fastest), and at
    the atoms: two-dielectric harmonic edge weights at the surface crossings, lumped
    screening mass, trilinear charges, screened Coulomb values on the box faces."""
    kT = 1.380649e-23 * spec.physics.T
    e, e0, ang = 1.602176634e-19, 8.85418781762e-12, 1e-10
    unit = 4.0 * math.pi * e0 * kT * ang / (e * e)
    eps_in, eps_out = unit * spec.physics.e_in, unit * spec.physics.e_out
    k2 = 2.0 * 1.0e3 * 6.022e23 * spec.physics.ionic_strength * ang**2 * e * e / (e0 * spec.physics.e_out * kT)
    n, h = int(spec.n[0]) + 1, spec.hf
    xyz, r = torch.from_numpy(atoms.xyz).to(device), torch.from_numpy(atoms.r).to(device)
    q = torch.from_numpy(atoms.q).to(device)
    c = [float(spec.origin[d]) + torch.arange(n, dtype=torch.float64, device=device) * h for d in range(3)]
    inside = torch.zeros(n, n, n, dtype=torch.bool, device=device)  # [z, y, x]
    bnd = torch.zeros(n, n, n, dtype=torch.float64, device=device)
    for a in range(atoms.n):
        d2 = ((c[2] - xyz[a, 2]) ** 2)[:, None, None] + ((c[1] - xyz[a, 1]) ** 2)[None, :, None] \
            + ((c[0] - xyz[a, 0]) ** 2)[None, None, :]
        inside |= d2 < r[a] ** 2
        d = d2.sqrt_()
        bnd += q[a] * torch.exp(-math.sqrt(k2) * d) / (d * eps_out)
    eps = torch.full_like(bnd, eps_out).masked_fill_(inside, eps_in)
    cond = []
    for axis, dim in ((2, 0), (1, 1), (0, 2)):  # z, y, x edges along tensor dimensions 0, 1, 2
        i1, i2 = inside.narrow(dim, 0, n - 1), inside.narrow(dim, 1, n - 1)
        e1, e2 = eps.narrow(dim, 0, n - 1), eps.narrow(dim, 1, n - 1)
        f = torch.full_like(e1, 0.5)
        at = (i1 != i2).nonzero()
        if at.numel():
            o = [d for d in range(3) if d != axis]
            co = lambda d: c[d][at[:, 2 - d]]
            t = _crossings(co(o[0]), co(o[1]), xyz, r, axis, co(axis), co(axis) + h, i2[i1 != i2])
            f[i1 != i2] = (t - co(axis)) / h
        cond.append(h / (f / e1 + (1.0 - f) / e2))
    i = slice(1, -1)
    lo = [cond[0][:-1, i, i], cond[1][i, :-1, i], cond[2][i, i, :-1]]
    hi = [cond[0][1:, i, i], cond[1][i, 1:, i], cond[2][i, i, 1:]]
    diag = sum(lo) + sum(hi) + (~inside).double()[i, i, i] * (eps_out * k2 * h**3)
    rhs = torch.zeros(n, n, n, dtype=torch.float64, device=device)
    u = [(xyz[:, d] - float(spec.origin[d])) / h for d in range(3)]
    base = [v.floor().long().clamp(0, n - 2) for v in u]
    corners = []
    for k in range(8):
        w = torch.ones_like(q)
        at = []
        for d in range(3):
            b = (k >> d) & 1
            f = u[d] - base[d]
            w = w * (f if b else 1.0 - f)
            at.append(base[d] + b)
        corners.append((at, w))
        rhs.index_put_((at[2], at[1], at[0]), 4.0 * math.pi * q * w, accumulate=True)
    phi = bnd.clone()
    phi[i, i, i] = 0.0
    b = rhs[i, i, i].clone()
    for a in range(3):  # known boundary neighbours move to the right-hand side
        m = n - 2
        b.narrow(a, 0, 1).add_(lo[a].narrow(a, 0, 1) * phi.narrow(a, 0, 1)[tuple(slice(None) if d == a else i for d in range(3))])
        b.narrow(a, m - 1, 1).add_(hi[a].narrow(a, m - 1, 1) * phi.narrow(a, n - 1, 1)[tuple(slice(None) if d == a else i for d in range(3))])
    phi[i, i, i] = _cg(lo, hi, diag, b)
    at_atoms = sum(phi[at[2], at[1], at[0]] * w for at, w in corners)
    return phi.reshape(-1), at_atoms


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "csr":
        lo, hi, diag, rhs = _blob(case["m"], seed, device)
        return _cg(lo, hi, diag, rhs).reshape(-1)
    if kind in ("request", "step") and case.get("grid"):
        spec = _reference(case)
        phi, at = _uniform(spec, _snapshot(spec, seed), device)
        out = {"phi": phi, "polar": None, "ionic": None}
        return dict(out, at_atoms=at) if kind == "request" else out
    if kind == "batch" and case["systems"] <= 12:
        phi = [_uniform(s, s.atoms, device)[0] for s in _batch_specs(case, seed)]
        return {"phi": torch.cat(phi), "energies": None}
    if kind == "outputs":  # Coulomb potential and field of the other atoms, and their energy
        spec = _reference(case)
        a = _snapshot(spec, seed)
        xyz, q = torch.from_numpy(a.xyz).to(device), torch.from_numpy(a.q).to(device)
        kT = 1.380649e-23 * spec.physics.T
        eps = 4.0 * math.pi * 8.85418781762e-12 * spec.physics.e_in * kT * 1e-10 / 1.602176634e-19**2
        d = xyz[:, None] - xyz[None]
        r = (d**2).sum(2).sqrt()
        r.fill_diagonal_(torch.inf)
        pot = (q / r).sum(1) / eps
        field = (d * (q / r**3)[:, :, None]).sum(1) / eps
        return {"coulomb": torch.cat([pot[:, None], field], 1), "surface": None, "at_atoms": None, "polar": None,
                "ionic": None, "coulomb_energy": 0.5 * float((q * pot).sum())}
    return None  # adaptive meshes and analytic molecular surfaces have no short 64-bit form
