"""Timed cases of the H.psi / Davidson / density path: what is timed, on which inputs, and the
64-bit values of the outputs that have one.

A case is one call through the public entry points, on silicon cells with the norm-conserving
PBE dataset of this package:

* ``apply``         H|psi> of a block of bands at one k-point (``Hamiltonian.apply``) or of the
                    whole k-batch in one launch per kernel (``Hamiltonian.apply_batched``):
                    what every eigensolver step spends its time on. Sphere -> grid transform,
                    V_eff, grid -> sphere transform, kinetic term and projector products.
* ``density``       ``compute_density`` over the occupied bands: once per SCF step.
* ``orthogonalize`` ``orthogonalize_against``: the new Davidson directions against the subspace.
* ``scf``           ``run_scf`` stopped after a fixed number of density updates: the whole call.

Cells are ``r1 x r2 x r3`` conventional diamond cells (8 atoms each, ``"cubic"``) or the 2-atom
primitive cell (``"fcc"``), with seeded displacements; unequal repeats give non-cubic FFT grids.
Everything a call needs beforehand (system, projector tables, bands, potential) is made from the
seed on the GPU.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from amaterasu_amd import Hamiltonian, compute_density
from amaterasu_amd.basis import FFTGrid, GSphere
from amaterasu_amd.eigen import orthogonalize_against
from amaterasu_amd.pseudo import Projectors, radial_form_factor
from amaterasu_amd.scf import SCFSettings, run_scf
from amaterasu_amd.system import DeviceSystem, KPoints, attach_ionic_fields, build_system, load_dataset

BOHR_IN_ANG = 0.5291772105638411
A0 = 5.431 / BOHR_IN_ANG
DIAMOND = np.array([[0.0, 0.0, 0.0], [0.0, 0.5, 0.5], [0.5, 0.0, 0.5], [0.5, 0.5, 0.0],
                    [0.25, 0.25, 0.25], [0.25, 0.75, 0.75], [0.75, 0.25, 0.75], [0.75, 0.75, 0.25]])
CHANNELS_PER_ATOM = 18  # projector rows of one Si atom: two radial channels each of l = 0, 1, 2


# ----------------------------------------------------------------------------- cases
def _case(kind, cell, r1, r2, r3, ecut, nk, bands, precision, **more):
    return {"kind": kind, "cell": cell, "r1": r1, "r2": r2, "r3": r3, "ecut": float(ecut), "nk": nk,
            "bands": bands, "precision": precision, "vacancies": 0, **more}


def listed():
    return [
        # the 2-atom cell, 8 bands at one k-point (28^3 grid): the smallest call, bound by launches
        {"name": "si2-apply-fp64", **_case("apply", "fcc", 1, 1, 1, 15, 1, 8, "fp64")},
        # the kernel-level batch: 16 ragged k-points of 64 bands each (42^3), in both precisions
        {"name": "si8-kbatch-fp32", **_case("apply", "cubic", 1, 1, 1, 20, 16, 64, "fp32")},
        {"name": "si8-kbatch-fp64", **_case("apply", "cubic", 1, 1, 1, 20, 16, 64, "fp64")},
        # an elongated cell: a non-cubic grid (42 x 42 x 84), the block of one small k-mesh
        {"name": "si16-tetragonal-fp64", **_case("apply", "cubic", 1, 1, 2, 20, 4, 40, "fp64")},
        # the 64-atom supercell at Gamma (84^3): a full block of bands, in both precisions
        {"name": "si64-apply-fp32", **_case("apply", "cubic", 2, 2, 2, 20, 1, 160, "fp32")},
        {"name": "si64-apply-fp64", **_case("apply", "cubic", 2, 2, 2, 20, 1, 160, "fp64")},
        # the largest cell (3x3x3 with two vacancies, 108^3): a full block in FP32, and in FP64 the
        # new directions of a step, where most bands have converged (an odd number of them)
        {"name": "si214-apply-fp32", **_case("apply", "cubic", 3, 3, 3, 15, 1, 440, "fp32", vacancies=2)},
        {"name": "si214-apply-fp64", **_case("apply", "cubic", 3, 3, 3, 15, 1, 45, "fp64", vacancies=2)},
        # the density of the occupied bands of the 64-atom cell
        {"name": "si64-density-fp64", **_case("density", "cubic", 2, 2, 2, 20, 1, 160, "fp64")},
        # 160 new directions against a 480-row subspace, as a Davidson step of the 64-atom cell does
        {"name": "si64-orthogonalize-fp32", **_case("orthogonalize", "cubic", 2, 2, 2, 20, 1, 160, "fp32", basis=480)},
        # whole calls: two SCF steps of the 64-atom cell at Gamma, and six of the 8-atom cell on
        # the time-reversal-reduced shifted 2x2x2 mesh (k-batched)
        {"name": "si64-scf-fp64", **_case("scf", "cubic", 2, 2, 2, 20, 1, 160, "fp64", steps=2)},
        {"name": "si8-scf-fp64", **_case("scf", "cubic", 1, 1, 1, 15, 4, 20, "fp64", steps=6)},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50.0)


def draw(rng):
    """One case of the same ranges: cells from 2 to 216 atoms (cubic and not), cutoffs 8-22 Ha
    (grid lengths 20-108, ecut 8-15 for the largest), 1-16 k-points, 1-440 bands per k-point in
    blocks of any size."""
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["apply"] * 6 + ["density"] * 2 + ["orthogonalize"] * 2 + ["scf"])
        precision = rng.choice(["fp32", "fp64"])
        more = {}
        if rng.random() < 0.2 and kind != "scf":
            cell, r, ecut, natoms = "fcc", (1, 1, 1), rng.uniform(8, 22), 2
        else:
            cell = "cubic"
            r = rng.choice([(1, 1, 1), (1, 1, 1), (1, 1, 2), (2, 1, 1), (1, 2, 2), (2, 2, 1), (2, 2, 2), (2, 2, 2),
                            (1, 1, 3), (3, 3, 3)])
            natoms = 8 * r[0] * r[1] * r[2]
            ecut = rng.uniform(8, 15) if r == (3, 3, 3) else rng.uniform(8, 22)
        ecut = round(ecut, 2)
        full = max(8, int(round(2.4 * natoms)))  # the bands of an SCF at this size
        nk = 1 if natoms >= 64 else _log_int(rng, 1, 16)
        bands = min(440, _log_int(rng, 1 if kind == "apply" else 4, 2 * full))
        if kind == "density":
            precision = "fp64"
        elif kind == "orthogonalize":
            nk, more = 1, {"basis": full * rng.choice([1, 2, 3])}
            bands = min(bands, full)
        elif kind == "scf":
            if natoms > 64:
                continue
            precision, nk, bands = "fp64", rng.choice([1, 2, 4]) if natoms < 64 else 1, full
            ecut = round(min(ecut, 20.0 if natoms < 64 else 16.0), 2)
            more = {"steps": rng.choice([1, 2])}
        case = _case(kind, cell, *r, ecut, nk, bands, precision, **more)
        if bands + more.get("basis", 0) <= 0.2 * _npw(case) and _cost(case) <= limit:
            return case


# ----------------------------------------------------------------------------- inputs
def _geometry(case, rng):
    if case["cell"] == "fcc":
        cell = 0.5 * A0 * np.array([[0.0, 1.0, 1.0], [1.0, 0.0, 1.0], [1.0, 1.0, 0.0]])
        frac = np.array([[0.0, 0.0, 0.0], [0.25, 0.25, 0.25]])
    else:
        r = np.array([case["r1"], case["r2"], case["r3"]])
        cell = np.diag(A0 * r)
        shifts = np.stack(np.meshgrid(*[np.arange(n) for n in r], indexing="ij"), axis=-1).reshape(-1, 3)
        frac = ((DIAMOND[None] + shifts[:, None]) / r).reshape(-1, 3)
    pos = frac @ cell
    pos = pos + rng.normal(scale=0.05 / BOHR_IN_ANG, size=pos.shape)
    if case["vacancies"]:
        pos = np.delete(pos, rng.choice(len(pos), size=case["vacancies"], replace=False), axis=0)
    return cell, pos


def _kpoints(case):
    """Gamma for one k-point of a supercell; else scattered points (the same for every seed: they
    fix the shapes), whose plane-wave counts are spread by up to +-8 % through a per-k cutoff, as
    in the kernel-level batch."""
    nk = case["nk"]
    rng = np.random.default_rng([2024, nk])
    if nk == 1:
        return np.zeros((1, 3)) if case["cell"] == "cubic" else np.full((1, 3), 0.25), np.array([case["ecut"]])
    d = rng.uniform(-0.08, 0.08, size=nk)
    return rng.uniform(-0.5, 0.5, size=(nk, 3)), case["ecut"] * (1.0 + d) ** (2.0 / 3.0)


@functools.lru_cache(maxsize=4)
def _radial_tables(qmax):
    """The dataset's projector form factors on a fine |q| mesh: (mesh step, channels, tables)."""
    ds = load_dataset()
    q = np.linspace(0.0, qmax, 1500)
    return q[1], [(c.l, c.energy) for c in ds.projectors], [radial_form_factor(ds, c, q) for c in ds.projectors]


def _interpolate(table, step, q):
    """Four-point Lagrange interpolation of an even function of q tabulated at 0, step, ..."""
    t = torch.as_tensor(table, device=q.device)
    x = q / step
    i = x.floor().long().clamp(1, len(t) - 3)
    u = x - i
    return (t[i - 1] * (-u * (u - 1) * (u - 2) / 6) + t[i] * ((u + 1) * (u - 1) * (u - 2) / 2)
            + t[i + 1] * (-(u + 1) * u * (u - 2) / 2) + t[i + 2] * ((u + 1) * u * (u - 1) / 6))


def _harmonics(l, v):
    n = torch.linalg.vector_norm(v, dim=1).clamp_min(1e-14)
    x, y, z = (v / n[:, None]).T
    if l == 0:
        return [torch.full_like(x, 0.5 / math.sqrt(math.pi))]
    if l == 1:
        c = math.sqrt(0.75 / math.pi)
        return [c * y, c * z, c * x]
    c = 0.5 * math.sqrt(15.0 / math.pi)
    return [c * x * y, c * y * z, 0.25 * math.sqrt(5.0 / math.pi) * (3 * z * z - 1), c * x * z, 0.5 * c * (x * x - y * y)]


def _projectors(sphere, pos, volume, qmax):
    """Kleinman-Bylander tables of one sphere, the form factors interpolated in |k+G|."""
    kg = torch.as_tensor(np.asarray(sphere.cartesian, dtype=float), device="cuda")
    q = torch.linalg.vector_norm(kg, dim=1)
    step, channels, tables = _radial_tables(qmax)
    rows, ls, cs, energies = [], [], [], []
    for c, ((l, energy), table) in enumerate(zip(channels, tables)):
        f = _interpolate(table, step, q) * (4.0 * math.pi / math.sqrt(volume))
        for m, y in enumerate(_harmonics(l, kg)):
            rows.append((-1j) ** l * (f * y))
            ls.append(l), cs.append((c, m - l)), energies.append(energy)
    rows = torch.stack(rows)
    p = torch.as_tensor(pos, device="cuda")
    matrix = torch.empty((len(p) * len(rows), len(q)), dtype=torch.complex128, device="cuda")
    for a in range(len(p)):
        matrix[a * len(rows):(a + 1) * len(rows)] = rows * torch.exp(-1j * (kg @ p[a]))
    dij = np.diag(np.tile(np.array(energies), len(p)))
    labels = [(a, l, c, m) for a in range(len(p)) for l, (c, m) in zip(ls, cs)]
    return Projectors(matrix=matrix, dij=dij, labels=labels)


def _system(case, seed, projectors=True):
    rng = np.random.default_rng([seed, 1])
    cell, pos = _geometry(case, rng)
    points, ecuts = _kpoints(case)
    grid = FFTGrid.for_cutoff(cell, 4.0 * case["ecut"])
    spheres = [GSphere.build(cell, float(e), kpoint=k) for e, k in zip(ecuts, points)]
    qmax = 1.05 * math.sqrt(2.0 * case["ecut"] * 1.08)
    proj = [_projectors(s, pos, grid.volume, qmax) for s in spheres] if projectors else None
    return DeviceSystem(cell=cell, positions=pos, symbols=["Si"] * len(pos), grid=grid, wave_spheres=spheres,
                        projectors=proj, kpoints=KPoints(points, np.full(len(points), 1.0 / len(points))), nspin=1,
                        nbands=case["bands"], nelectrons=4.0 * len(pos), ecut_rho=4.0 * case["ecut"])


def _potential(shape, gen, sigma=2.0):
    """A smooth real field of 1 Ha RMS: normal noise under a periodic Gaussian of two grid cells."""
    v = torch.randn(shape, dtype=torch.float64, device="cuda", generator=gen)
    m2 = sum((torch.fft.fftfreq(n, device="cuda", dtype=torch.float64) ** 2).reshape([-1 if a == b else 1 for b in range(3)])
             for a, n in enumerate(shape))
    v = torch.fft.ifftn(torch.fft.fftn(v) * torch.exp(-2.0 * math.pi**2 * sigma**2 * m2)).real
    v = v - v.mean()
    return (v / v.square().mean().sqrt()).contiguous()


def _normal(gen, *shape):
    return torch.randn(shape, dtype=torch.complex128, device="cuda", generator=gen)


def _g2(sphere):
    return torch.as_tensor(np.asarray(sphere.g2, dtype=float), device="cuda")


def _bands(system, nbands, gen):
    """Seeded coefficients falling off as 1/(1 + |k+G|^2)^2, normalised: [nk][nbands][widest k],
    zero past each k-point's own plane waves."""
    wide = max(len(s.g2) for s in system.wave_spheres)
    out = torch.zeros((len(system.wave_spheres), nbands, wide), dtype=torch.complex128, device="cuda")
    for k, s in enumerate(system.wave_spheres):
        c = _normal(gen, nbands, len(s.g2)) / (1.0 + _g2(s)) ** 2
        out[k, :, : len(s.g2)] = c / torch.linalg.vector_norm(c, dim=1, keepdim=True)
    return out


def _orthonormal(block):
    for _ in range(2):
        low = torch.linalg.cholesky(block @ block.mH)
        block = torch.linalg.solve_triangular(low, torch.eye(len(low), dtype=low.dtype, device="cuda"), upper=False) @ block
    return block


def _dtype(case):
    return torch.complex64 if case["precision"] == "fp32" else torch.complex128


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return gen


def _scf_system(case, seed):
    rng = np.random.default_rng([seed, 1])
    cell, pos = _geometry(case, rng)
    mesh = np.array([[0.25, 0.25, 0.25], [0.25, 0.25, -0.25], [0.25, -0.25, 0.25], [-0.25, 0.25, 0.25]])
    points = np.zeros((1, 3)) if case["nk"] == 1 else mesh[: case["nk"]]
    ds = load_dataset()
    system = build_system(cell, pos, ["Si"] * len(pos), {"Si": ds}, 4.0 * case["ecut"], points, case["ecut"],
                          nbands=case["bands"])
    return attach_ionic_fields(system, {"Si": ds}, 4.0 * case["ecut"], xc="PBE")


def prepare(case, seed):
    state = {"case": case}
    gen = _generator(seed)
    if case["kind"] == "scf":
        system = state["system"] = _scf_system(case, seed)
        state["density"] = system.initial_density()
        state["settings"] = SCFSettings(max_steps=case["steps"], tol_energy=1e-12, tol_density=1e-12)
        return state
    system = state["system"] = _system(case, seed, projectors=case["kind"] == "apply")
    if case["kind"] == "apply":
        state["psi"] = _bands(system, case["bands"], gen).to(_dtype(case))
        state["potential"] = _potential(system.grid.shape, gen)
        state["hamiltonian"] = Hamiltonian(system, state["potential"], precision=case["precision"])
    elif case["kind"] == "density":
        psi = _bands(system, case["bands"], gen).to(_dtype(case))
        state["bands"] = [[psi[k, :, : len(s.g2)].contiguous() for k, s in enumerate(system.wave_spheres)]]
        occ = np.ones((1, case["nk"], case["bands"]))
        occ[:, :, math.ceil(0.8 * case["bands"]):] = 0.0  # the empty bands of the block
        state["occupations"] = occ
    else:
        t = 0.5 * _g2(system.wave_spheres[0])
        basis = _orthonormal(_normal(gen, case["basis"], len(t)) / (1.0 + t))
        new = _normal(gen, case["bands"], len(t)) / (1.0 + t * t)
        new = new + _normal(gen, case["bands"], case["basis"]) / math.sqrt(case["basis"]) @ basis
        state["basis"] = basis.to(_dtype(case))
        state["block"] = (new / torch.linalg.vector_norm(new, dim=1, keepdim=True)).to(_dtype(case))
    return state


# ----------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    if case["kind"] == "apply":
        h = state["hamiltonian"]
        return h.apply_batched(state["psi"]) if case["nk"] > 1 else h.apply(state["psi"][0], 0)
    if case["kind"] == "density":
        return compute_density(state["system"], state["bands"], state["occupations"], device=True)
    if case["kind"] == "orthogonalize":
        return orthogonalize_against(state["block"], state["basis"])
    r = run_scf(state["system"], state["settings"], density=state["density"])
    return {"density": r.density, "eigenvalues": r.eigenvalues, "occupations": r.occupations,
            "energy": r.energies.total}


# ----------------------------------------------------------------------------- work
def _natoms(case):
    return 2 if case["cell"] == "fcc" else 8 * case["r1"] * case["r2"] * case["r3"] - case["vacancies"]


def _volume(case):
    return A0**3 * (0.25 if case["cell"] == "fcc" else case["r1"] * case["r2"] * case["r3"])


def _npw(case):
    return _volume(case) * (2.0 * case["ecut"]) ** 1.5 / (6.0 * math.pi**2)


def _ngrid(case):
    """Points of a grid that holds the density's sphere, of twice the bands' radius."""
    return _volume(case) * (2.0 * case["ecut"]) ** 1.5 * 8.0 / math.pi**3


def _apply_work(case, bands):
    """One H|psi> block: bands in and out, the potential and the projector table once; the FFT
    pair pruned to the sphere (all columns along one axis, half and a fifth along the others),
    and the two projector products."""
    s = 8 if case["precision"] == "fp32" else 16
    npw, nproj, n = _npw(case), CHANNELS_PER_ATOM * _natoms(case), _ngrid(case)
    logs = 1.7 * math.log2(n) / 3.0
    total = bands * case["nk"]
    return {"bytes": 2.0 * total * npw * s + n * s / 2 + case["nk"] * nproj * npw * s,
            "flops": total * (2 * 5.0 * n * logs + 2.0 * n + 16.0 * npw * nproj)}


def work(case):
    npw, nb, nk = _npw(case), case["bands"], case["nk"]
    s = 8 if case["precision"] == "fp32" else 16
    one = _apply_work(case, nb)
    n = _ngrid(case)
    if case["kind"] == "apply":
        return one
    if case["kind"] == "density":
        occ = math.ceil(0.8 * nb) * nk
        return {"bytes": occ * npw * s + 8.0 * n, "flops": occ * (5.0 * n * 1.7 * math.log2(n) / 3.0 + 4.0 * n)}
    if case["kind"] == "orthogonalize":
        # two projections off the basis (overlap and update each), one orthonormalisation
        return {"bytes": (case["basis"] + 2.0 * nb) * npw * s,
                "flops": 8.0 * npw * nb * (4.0 * case["basis"] + 2.0 * nb)}
    # Davidson steps of nb new directions each over a subspace that cycles through 2, 3 and 4 nb rows:
    # H on them, two projections and an orthonormalisation, the new columns of the projected
    # matrix, two rotations, and the eigensolve of the projected matrix
    steps = (40 + 20 * (case["steps"] - 1)) * nk
    m = 3.0 * nb
    flops = one["flops"] / nk + 8.0 * npw * nb * (4.0 * m + 2.0 * nb + m + 2.0 * m) + 16.0 / 3.0 * m**3
    return {"bytes": steps * (one["bytes"] / nk + 3.0 * m * npw * s), "flops": steps * flops}


# ----------------------------------------------------------------------------- 64-bit values
def _flat_index(sphere, shape):
    h = np.mod(np.asarray(sphere.miller), np.array(shape))
    return torch.as_tensor(np.ravel_multi_index(tuple(h.T), shape).astype(np.int64), device="cuda")


def _to_real(rows, flat, shape):
    """u(r) = sum_G c_G e^{iGr} of a few rows."""
    grid = torch.zeros((len(rows), math.prod(shape)), dtype=torch.complex128, device="cuda")
    grid[:, flat] = rows
    return torch.fft.ifftn(grid.reshape(-1, *shape), dim=(1, 2, 3), norm="forward")


def exact(case, seed):
    if case["kind"] == "scf":  # an iteration that has not converged: no value of its own
        return None
    state = prepare(case, seed)
    system = state["system"]
    shape = tuple(system.grid.shape)
    chunk = max(1, int(2e9 // (16 * math.prod(shape))))
    if case["kind"] == "apply":
        out = torch.zeros(state["psi"].shape, dtype=torch.complex128, device="cuda")
        for k, (s, p) in enumerate(zip(system.wave_spheres, system.projectors)):
            flat, npw, g2 = _flat_index(s, shape), len(s.g2), _g2(s)
            dij = torch.as_tensor(np.diag(p.dij).copy(), device="cuda")
            for b in range(0, case["bands"], chunk):
                c = state["psi"][k, b:b + chunk, :npw].to(torch.complex128)
                u = _to_real(c, flat, shape) * state["potential"]
                h = torch.fft.fftn(u, dim=(1, 2, 3), norm="forward").reshape(len(c), -1)[:, flat] + 0.5 * g2 * c
                out[k, b:b + chunk, :npw] = h + ((c @ p.matrix.mH) * dij) @ p.matrix
        return out if case["nk"] > 1 else out[0]
    if case["kind"] == "density":
        rho = torch.zeros((1, *shape), dtype=torch.float64, device="cuda")
        for k, s in enumerate(system.wave_spheres):
            flat = _flat_index(s, shape)
            rows = np.flatnonzero(state["occupations"][0, k])
            for b in range(0, len(rows), chunk):
                u = _to_real(state["bands"][0][k][b:min(b + chunk, len(rows))].to(torch.complex128), flat, shape)
                rho[0] += (2.0 / case["nk"] / system.grid.volume) * (u.real**2 + u.imag**2).sum(0)
        return rho
    b, q = state["block"].to(torch.complex128), state["basis"].to(torch.complex128)
    for _ in range(2):
        b = b - (b @ q.mH) @ q
    return _orthonormal(b)
