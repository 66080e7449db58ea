"""Density accumulation on the GPU against the oracle's compute_density (scf/density.py:35-84)."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_density_matches_oracle(si2_system):
    from amaterasu_amd.density import compute_density, electron_count
    from oracle.density import compute_density as ocd
    from oracle.eigen import random_bands

    s = si2_system
    wf = [[random_bands(len(sp), s.nbands, sp.kinetic_energy, seed=7 + ik) for ik, sp in enumerate(s.wave_spheres)]]
    occ = np.zeros((1, 2, s.nbands))
    occ[:, :, :4] = 1.0
    occ[0, 1, 4] = 0.3  # a fractional occupation
    occ[0, 0, 5] = 1e-13  # below the 1e-12 activity cut (density.py:64-67)
    got, ref = compute_density(s, wf, occ), ocd(s, wf, occ)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-12
    assert electron_count(s, got) == pytest.approx(8.0 + 2 * 0.75 * 0.3, abs=1e-9)


def test_density_fp32_orbitals(si2_system):
    import torch

    from amaterasu_amd.density import compute_density
    from oracle.density import compute_density as ocd
    from oracle.eigen import random_bands

    s = si2_system
    wf = [[random_bands(len(sp), s.nbands, sp.kinetic_energy, seed=ik) for ik, sp in enumerate(s.wave_spheres)]]
    occ = np.zeros((1, 2, s.nbands))
    occ[:, :, :4] = 1.0
    wf32 = [[torch.from_numpy(w).to("cuda", torch.complex64) for w in wf[0]]]
    got, ref = compute_density(s, wf32, occ), ocd(s, wf, occ)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-5


def test_density_generic_grid(si2_system):
    """Non-cubic grid: the generic density kernels against the oracle."""
    import copy

    from amaterasu_amd.density import compute_density
    from oracle.basis import FFTGrid
    from oracle.density import compute_density as ocd
    from oracle.eigen import random_bands

    s = copy.copy(si2_system)
    s.grid = FFTGrid((24, 20, 22), si2_system.cell)
    wf = [[random_bands(len(sp), s.nbands, sp.kinetic_energy, seed=3 + ik) for ik, sp in enumerate(s.wave_spheres)]]
    occ = np.zeros((1, 2, s.nbands))
    occ[:, :, :5] = 0.8
    got, ref = compute_density(s, wf, occ), ocd(s, wf, occ)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-12


@pytest.mark.parametrize("shape", [(1, 1), (2, 255), (1, 257), (2, 65537), (3, 200000)])
@pytest.mark.parametrize("kind", ["mixed", "zero", "negative", "nan"])
def test_finish_density(shape, kind):
    """Division, floor and rescaling per spin against the formula: a sum over n numbers of
    size 1 errs by at most n u of the sum of sizes, relative to a kept sum of at least a third of it."""
    import torch

    from amaterasu_amd import ops

    rng = np.random.default_rng(shape[1])
    x = rng.normal(size=shape) + 0.8
    if kind == "zero":
        x[:] = 0.0
    elif kind == "negative":
        x = -np.abs(x)
    elif kind == "nan":
        x[0, -1] = np.nan
    v = 3.7
    y = x / v
    kept = np.where(y < 0, 0.0, y)
    before, after = y.sum(1), kept.sum(1)
    with np.errstate(invalid="ignore", divide="ignore"):
        scale = np.where(after > 0, before / np.where(after > 0, after, 1.0), 1.0)
    want = kept * scale[:, None]
    got = ops.finish_density(torch.from_numpy(x.copy()).cuda(), v).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert (np.abs(got - want)[ok] <= 6 * shape[1] * 2.0**-53 * np.abs(kept).max(initial=0.0, where=ok) + 0.0).all()


@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("nlist", [1, 2, 3, 7, 12])
def test_density_chunk_choice(si2_system, nlist, dtype):
    """The chosen chunk sums the same squares as one band per chunk, in another order."""
    import torch

    from amaterasu_amd.hamiltonian import device_plan

    plan = device_plan(si2_system)
    psi = torch.randn(2, 6, plan.npw_pad, dtype=getattr(torch, dtype), device="cuda") / np.sqrt(plan.npw_pad)
    for k in range(2):
        psi[k, :, plan.npw[k] :] = 0
    rows = np.arange(nlist, dtype=np.int32)
    w = np.linspace(0.3, 1.7, nlist)
    chunk = plan.density_chunk(psi.dtype, nlist)
    assert 1 <= chunk <= max(nlist, 8)
    out = []
    for c in (chunk, 1):
        rho = torch.full(plan.shape, float("nan"), dtype=torch.float64, device="cuda")
        plan.accumulate_density(psi, rows, w, rho, beta=0.0, chunk=c)
        out.append(rho.cpu().numpy())
    assert np.abs(out[0] - out[1]).max() <= 2 * nlist * 2.0**-53 * np.abs(out[1]).max()


@pytest.mark.parametrize("n,bands,dtype,rounds", [(32, 64, "complex128", 1), (42, 40, "complex128", 1),
                                                  (28, 64, "complex128", 1), (25, 64, "complex128", 2),
                                                  (84, 128, "complex128", 1), (32, 64, "complex64", 1),
                                                  (44, 40, "complex64", 1), (42, 64, "complex64", 2)])
def test_chunk_counts_a_cu_shared_by_two_workgroups(n, bands, dtype, rounds):
    """Partial sums that one workgroup a CU can hold are not split over two (n planes times the chunks: at
    most 256 workgroups) where two in FP64, or in FP32 at the lengths 4 a, would wait for each other;
    other FP32 lengths and short odd FP64 ones gain from two."""
    import torch

    from amaterasu_amd.basis import GSphere
    from amaterasu_amd.device import DevicePlan

    sphere = GSphere.build(np.eye(3) * n / 4.0, 0.5 * ((n / 4.0 - 0.4) * 2.0 * np.pi / (n / 4.0)) ** 2)
    chunk = DevicePlan((n, n, n), [sphere]).density_chunk(getattr(torch, dtype), bands)
    assert 1 <= chunk <= bands and -(-(-(-bands // chunk) * n) // 256) == rounds
