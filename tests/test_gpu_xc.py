"""The device grid-side operators against the oracle on the Si2 grid: exchange-correlation
energies and potentials (LDA-PZ, LDA-PW, PBE, PBEsol; spin-unpolarised and polarised;
``xc/driver.py:108-164``) and the Hartree energy and potential (``hartree.py:28-50``)."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _density(shape, nspin, seed):
    rng = np.random.default_rng(seed)
    i, j, k = np.meshgrid(*[np.arange(n) / n for n in shape], indexing="ij")
    base = 0.05 + 0.04 * np.cos(2 * np.pi * (i + j)) ** 2 + 0.03 * np.sin(2 * np.pi * k) ** 2
    base = base + 0.002 * rng.random(shape)
    if nspin == 1:
        return base[None]
    return np.stack([0.6 * base, 0.4 * base])


@pytest.mark.parametrize("name", ["LDA-PZ", "LDA-PW", "PBE", "PBEsol"])
@pytest.mark.parametrize("nspin", [1, 2])
def test_xc_on_the_grid_matches_the_oracle(si2_system, name, nspin):
    import torch

    from amaterasu_amd.xc import GridOps, XCFunctional
    from oracle.xc import XCFunctional as OXC

    grid = si2_system.grid
    rho = _density(grid.shape, nspin, 3)
    e_ref, v_ref = OXC(name).evaluate_on_grid(rho, grid)
    e, v = XCFunctional(name).evaluate_on_grid(torch.from_numpy(rho).cuda(), GridOps(grid.shape, grid.cell))
    v = v.cpu().numpy()
    assert e == pytest.approx(e_ref, rel=1e-12)
    assert v.shape == v_ref.shape
    assert np.abs(v - v_ref).max() < 1e-11 * np.abs(v_ref).max()


def test_hartree_matches_the_oracle(si2_system):
    import torch

    from amaterasu_amd.scf import GridSide
    from oracle.scf import hartree

    rho = _density(si2_system.grid.shape, 1, 4)[0]
    e_ref, v_ref = hartree(si2_system.grid, si2_system.density_sphere, rho)
    e, v = GridSide(si2_system).hartree(torch.from_numpy(rho).cuda())
    assert e == pytest.approx(e_ref, rel=1e-12)
    assert np.abs(v.cpu().numpy() - v_ref).max() < 1e-12 * np.abs(v_ref).max()


@pytest.mark.parametrize("n", [1, 255, 257, 4099])
@pytest.mark.parametrize("name", ["PBE", "PBEsol"])
def test_gga_points_match_the_oracle(name, n):
    """The pointwise kernel against the oracle at single points: both are chains of some hundred
    FP64 operations, so ordinary densities agree to 1e-11 of each value plus 1e-11 of the exchange
    scale; points at the edges (empty spin, below the threshold, zero gradient, negative) to 1e-7, as
    the derivative by the polarisation is of size 1e8 there."""
    import torch

    from amaterasu_amd import ops
    from amaterasu_amd.xc import _GGA
    from oracle.xc import XCFunctional as OXC

    rng = np.random.default_rng(n)
    tot = 10.0 ** rng.uniform(-5, 1, n)
    z = rng.uniform(-0.95, 0.95, n)
    rho = np.stack([0.5 * tot * (1 + z), 0.5 * tot * (1 - z)], -1)
    s = rng.uniform(0.0, 3.0, (n, 2)) * rho ** (4 / 3) * 6
    sig = np.stack([s[:, 0] ** 2, rng.uniform(-1, 1, n) * s[:, 0] * s[:, 1], s[:, 1] ** 2], -1)
    edge = np.array([[0.3, 0.0], [0.0, 0.2], [0.0, 0.0], [1e-25, 1e-26], [-1e-3, 0.1], [0.1, 0.1], [-0.1, -0.2]])
    edge_sig = np.array([[0.1, 0.0, 0.0], [0.0, 0.0, 0.2], [0, 0, 0], [0, 0, 0], [0, 0, 0.1], [0, 0, 0], [0, 0, 0]])
    par = [_GGA[name.upper()][k] for k in ("kappa", "mu", "beta", "gamma")]
    for r, g, tol in ((rho, sig, 1e-11), (edge, edge_sig, 1e-7)):
        with np.errstate(all="ignore"):
            eps, v, vs = OXC(name).evaluate(r, g)
        want = np.stack([eps, v[:, 0], v[:, 1], vs[:, 0], vs[:, 1], vs[:, 2]])
        dev = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (r[:, 0], r[:, 1], g[:, 0], g[:, 1], g[:, 2])]
        got = ops.gga(*dev, par).cpu().numpy()
        scale = np.abs(want)
        scale[:3] += np.maximum(r.sum(1), 0.0) ** (1 / 3)
        assert (np.abs(got - want) <= tol * scale).all()
