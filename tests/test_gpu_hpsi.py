"""H.psi on the GPU against the oracle's Hamiltonian.apply (hamiltonian/operator.py:60-69).

FP64 must match to ~1e-12 relative (summation order differs in the FFTs and GEMMs);
FP32 is reported against FP64 with a stated bound."""

from __future__ import annotations

import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _block(n, nb, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(nb, n)) + 1j * rng.normal(size=(nb, n))


def test_apply_matches_oracle_si2(si2_system):
    from amaterasu_amd.hamiltonian import Hamiltonian
    from oracle.hamiltonian import Hamiltonian as OH

    rng = np.random.default_rng(0)
    v = rng.normal(size=(1, *si2_system.grid.shape))
    h, o = Hamiltonian(si2_system, v), OH(si2_system, v)
    for ik in range(2):
        c = _block(len(si2_system.wave_spheres[ik]), 5, ik)
        got, ref = h.apply(c, ik), o.apply(c, ik)
        assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-12
        one = h.apply(c[2], ik)  # a single band (1-D) keeps its shape
        assert one.shape == c[2].shape and np.abs(one - ref[2]).max() / np.abs(ref).max() < 1e-12


def test_apply_generic_grid_matches_oracle(si2_system):
    """A non-cubic grid runs the generic (runtime-radix) kernels instead of the
    compile-time-length ones; both must agree with the oracle."""
    from amaterasu_amd.hamiltonian import Hamiltonian
    from oracle.basis import FFTGrid
    from oracle.hamiltonian import Hamiltonian as OH

    s = copy.copy(si2_system)
    s.grid = FFTGrid((24, 20, 22), si2_system.cell)
    rng = np.random.default_rng(11)
    v = rng.normal(size=(1, *s.grid.shape))
    h, o = Hamiltonian(s, v), OH(s, v)
    assert not h.plan.info[0] == h.plan.info[1] == h.plan.info[2]
    for ik in range(2):
        c = _block(len(s.wave_spheres[ik]), 3, 20 + ik)
        got, ref = h.apply(c, ik), o.apply(c, ik)
        assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-12
        got32 = Hamiltonian(s, v, precision="fp32").apply(c, ik)
        assert np.abs(got32 - ref).max() / np.abs(ref).max() < 5e-6


def test_apply_is_hermitian(si2_system):
    from amaterasu_amd.hamiltonian import Hamiltonian

    rng = np.random.default_rng(1)
    h = Hamiltonian(si2_system, rng.normal(size=(1, *si2_system.grid.shape)))
    b = _block(len(si2_system.wave_spheres[1]), 4, 2)
    m = b.conj() @ h.apply(b, 1).T
    assert np.abs(m - m.conj().T).max() < 1e-11


def test_wrong_potential_shape(si2_system):
    from amaterasu_amd.hamiltonian import Hamiltonian

    with pytest.raises(ValueError, match="effective potential has shape"):
        Hamiltonian(si2_system, np.zeros((2, *si2_system.grid.shape)))


def test_fp32_apply_error_is_bounded(si2_system):
    from amaterasu_amd.hamiltonian import Hamiltonian
    from oracle.hamiltonian import Hamiltonian as OH

    rng = np.random.default_rng(3)
    v = rng.normal(size=(1, *si2_system.grid.shape))
    c = _block(len(si2_system.wave_spheres[0]), 6, 4)
    ref = OH(si2_system, v).apply(c, 0)
    got = Hamiltonian(si2_system, v, precision="fp32").apply(c, 0)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 5e-6


def test_kbatch_matches_per_k_oracle(si_pseudo):
    """The ragged k-batch (padded [k][band][npw_pad] layout, one launch per kernel)
    against the oracle applied k by k, on 3 k-points of the Si8 kernel batch."""
    import torch

    from amaterasu_amd.hamiltonian import Hamiltonian
    from amaterasu_amd.system import build_system, load_dataset
    from amaterasu_amd.workloads import seeded_coefficients, si8_kbatch, smooth_potential
    from oracle.hamiltonian import Hamiltonian as OH
    from oracle.system import build_system as obuild

    spec = si8_kbatch(nk=3, nbands=6)
    sysd = build_system(spec.cell, spec.positions, spec.symbols, {"Si": load_dataset()}, spec.ecut_rho,
                        spec.kpoints, spec.ecuts)
    syso = obuild(spec.cell, spec.positions, spec.symbols, {"Si": si_pseudo}, float(spec.ecuts[0]), spec.ecut_rho,
                  spec.kpoints, wave_ecuts=spec.ecuts, with_ewald=False)
    assert sysd.grid.shape == syso.grid.shape == (42, 42, 42)
    v = smooth_potential(sysd.grid.shape, seed=spec.seed)
    hd = Hamiltonian(sysd, v)
    ho = OH(syso, v)
    plan = hd.plan
    psi = torch.zeros((3, 6, plan.npw_pad), dtype=torch.complex128, device="cuda")
    blocks = []
    for k, s in enumerate(sysd.wave_spheres):
        c = seeded_coefficients(s.g2, 6, seed=100 + k)
        blocks.append(c)
        psi[k, :, : len(s.g2)] = torch.from_numpy(c).cuda()
    out = hd.apply_batched(psi).cpu().numpy()
    for k, s in enumerate(sysd.wave_spheres):
        ref = ho.apply(blocks[k], k)
        got = out[k, :, : len(s.g2)]
        assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-12
        assert np.all(out[k, :, len(s.g2):] == 0)  # padding stays zero


def test_kbatch_fp32_band_pairs_across_k_points(si_pseudo):
    """FP32 k-batch on the 42^3 grid with an odd band count (5 bands at each of 3 k-points,
    so neighbouring band rows of the launch belong to different k-points, with different
    stick maps and row lists). Against the oracle k by k, at the FP32 bound of the
    single-k test."""
    import torch

    from amaterasu_amd.hamiltonian import Hamiltonian
    from amaterasu_amd.system import build_system, load_dataset
    from amaterasu_amd.workloads import seeded_coefficients, si8_kbatch, smooth_potential
    from oracle.hamiltonian import Hamiltonian as OH
    from oracle.system import build_system as obuild

    spec = si8_kbatch(nk=3, nbands=5)
    sysd = build_system(spec.cell, spec.positions, spec.symbols, {"Si": load_dataset()}, spec.ecut_rho,
                        spec.kpoints, spec.ecuts)
    syso = obuild(spec.cell, spec.positions, spec.symbols, {"Si": si_pseudo}, float(spec.ecuts[0]), spec.ecut_rho,
                  spec.kpoints, wave_ecuts=spec.ecuts, with_ewald=False)
    v = smooth_potential(sysd.grid.shape, seed=spec.seed)
    hd = Hamiltonian(sysd, v, precision="fp32")
    ho = OH(syso, v)
    plan = hd.plan
    psi = torch.zeros((3, 5, plan.npw_pad), dtype=torch.complex64, device="cuda")
    blocks = []
    for k, s in enumerate(sysd.wave_spheres):
        c = seeded_coefficients(s.g2, 5, seed=200 + k)
        blocks.append(c)
        psi[k, :, : len(s.g2)] = torch.from_numpy(c).to("cuda", torch.complex64)
    out = hd.apply_batched(psi).cpu().numpy()
    for k, s in enumerate(sysd.wave_spheres):
        ref = ho.apply(blocks[k], k)
        got = out[k, :, : len(s.g2)]
        assert np.abs(got - ref).max() / np.abs(ref).max() < 5e-6
        assert np.all(out[k, :, len(s.g2):] == 0)


def test_empty_lattice_free_electron_bands(si2_system):
    """Gate of test_hamiltonian.py:221-244 on the GPU path: V = 0, no projectors ->
    eigenvalues |k+G|^2/2 to 1e-11 Ha."""
    from amaterasu_amd.eigen import davidson, random_bands
    from amaterasu_amd.hamiltonian import Hamiltonian
    from oracle.pseudo import KBProjectors

    s = copy.copy(si2_system)
    s.projectors = [KBProjectors(np.zeros((0, len(sp)), dtype=complex), np.zeros((0, 0)), []) for sp in
                    s.wave_spheres]
    h = Hamiltonian(s, np.zeros((1, *s.grid.shape)))
    for ik, sp in enumerate(s.wave_spheres):
        r = davidson(lambda b, ik=ik: h.apply(b, ik), random_bands(len(sp), 10, sp.kinetic_energy, seed=ik),
                     sp.kinetic_energy, tolerance=1e-12, max_iterations=200)
        assert np.abs(r.eigenvalues - np.sort(sp.kinetic_energy)[:10]).max() < 1e-11


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_full_grid_route_matches_the_plane_kernels(si2_system, precision):
    """Grids whose (n2 x n3) plane does not fit one workgroup's LDS (FP64 planes above ~100^2,
    e.g. the 108^3 grid of Si214) take the full-grid route: the library's scatter, 3D
    transforms and gather. Forced here on the Si2 grid, it must give the pruned kernels' H.psi
    and density on the same inputs."""
    import torch

    from amaterasu_amd.device import DevicePlan
    from amaterasu_amd.ops import FP32, FP64

    s = si2_system
    plan = DevicePlan(s.grid.shape, s.wave_spheres, s.projectors)
    prec, dt = (FP64, torch.complex128) if precision == "fp64" else (FP32, torch.complex64)
    rng = np.random.default_rng(7)
    psi = torch.zeros((2, 6, plan.npw_pad), dtype=dt, device="cuda")
    for k in range(2):
        psi[k, :, : plan.npw[k]] = torch.from_numpy(_block(plan.npw[k], 6, 10 + k)).to(dt)
    v = torch.from_numpy(rng.normal(size=s.grid.shape)).cuda()
    rows, wts = np.arange(12), rng.uniform(0.1, 1.0, size=12)
    rho_a = torch.zeros(s.grid.shape, dtype=torch.float64, device="cuda")
    rho_b = torch.zeros_like(rho_a)
    ref = plan.hpsi(psi, v)
    plan.accumulate_density(psi, rows, wts, rho_a)
    plan.set_route(prec, True)
    assert not plan.plane_ok[prec]
    got = plan.hpsi(psi, v)
    plan.accumulate_density(psi, rows, wts, rho_b)
    tol = 1e-12 if precision == "fp64" else 2e-6
    assert (torch.abs(got - ref).max() / torch.abs(ref).max()).item() < tol
    assert (torch.abs(rho_b - rho_a).max() / rho_a.abs().max()).item() < tol


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_full_operator_entry_point_matches_the_call_sequence(si_pseudo, precision):
    """amt_hpsi (T + V_loc + V_NL in one call, projector tables attached to the plan with
    amt_plan_set_projectors) against the explicit sequence amt_hpsi_local, amt_zgemm (NC),
    amt_kb_dij, amt_zgemm (NN) through the C ABI on 3 ragged k-points of the Si8 batch:
    bit-identical, and a plan without tables gives the local part alone."""
    import torch

    from amaterasu_amd import ops
    from amaterasu_amd._lib import check, lib
    from amaterasu_amd.device import DevicePlan
    from amaterasu_amd.system import build_system, load_dataset
    from amaterasu_amd.workloads import seeded_coefficients, si8_kbatch, smooth_potential

    spec = si8_kbatch(nk=3, nbands=7)
    s = build_system(spec.cell, spec.positions, spec.symbols, {"Si": load_dataset()}, spec.ecut_rho, spec.kpoints,
                     spec.ecuts)
    plan = DevicePlan(s.grid.shape, s.wave_spheres, s.projectors)
    prec = 1 if precision == "fp64" else 0
    cdt = torch.complex128 if prec else torch.complex64
    psi = torch.zeros((3, 7, plan.npw_pad), dtype=cdt, device="cuda")
    for k, sp in enumerate(s.wave_spheres):
        psi[k, :, : len(sp.g2)] = torch.from_numpy(seeded_coefficients(sp.g2, 7, seed=40 + k)).to("cuda", cdt)
    v = torch.from_numpy(smooth_potential(s.grid.shape, seed=4)).to("cuda", ops.real_dtype(prec))
    mat, dij, start, length = plan.kb_tables(prec)
    stream = ops.stream_handle()
    # explicit sequence
    ref = torch.zeros_like(psi)
    st = plan.sticks(prec, 21)
    check(lib().amt_hpsi_local(plan.handle, prec, psi.data_ptr(), ref.data_ptr(), 7, 0, 3, v.data_ptr(),
                               st.data_ptr(), stream), "hpsi_local")
    local = ref.clone()
    proj = ops.zgemm(psi, mat, 1)
    pd = torch.empty_like(proj)
    check(lib().amt_kb_dij(prec, proj.data_ptr(), dij.data_ptr(), start.data_ptr(), length.data_ptr(), pd.data_ptr(),
                           7, plan.nproj, 7 * plan.nproj, plan.nproj * plan.nproj, 7 * plan.nproj, 3, stream), "kb_dij")
    ops.zgemm(pd, mat, 0, beta=1.0, out=ref)
    # one call
    check(lib().amt_plan_set_projectors(plan.handle, prec, plan.nproj, mat.data_ptr(), dij.data_ptr(),
                                        start.data_ptr(), length.data_ptr()), "plan_set_projectors")
    nbytes = lib().amt_hpsi_workspace(plan.handle, prec, 7, 3)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    got = torch.zeros_like(psi)
    check(lib().amt_hpsi(plan.handle, prec, psi.data_ptr(), got.data_ptr(), 7, 0, 3, v.data_ptr(), ws.data_ptr(),
                         nbytes, stream), "hpsi")
    torch.cuda.synchronize()
    assert torch.equal(got, ref)
    # a single k-point from the middle of the batch
    one = torch.zeros_like(psi[1:2])
    check(lib().amt_hpsi(plan.handle, prec, psi[1:2].data_ptr(), one.data_ptr(), 7, 1, 1, v.data_ptr(),
                         ws.data_ptr(), nbytes, stream), "hpsi")
    torch.cuda.synchronize()
    assert (torch.abs(one - ref[1:2]).max() / torch.abs(ref).max()).item() < (1e-14 if prec else 1e-6)
    # detached tables: the local part alone
    check(lib().amt_plan_set_projectors(plan.handle, prec, 0, None, None, None, None), "plan_set_projectors")
    bare = torch.zeros_like(psi)
    check(lib().amt_hpsi(plan.handle, prec, psi.data_ptr(), bare.data_ptr(), 7, 0, 3, v.data_ptr(), ws.data_ptr(),
                         nbytes, stream), "hpsi")
    torch.cuda.synchronize()
    assert torch.equal(bare, local)
    with pytest.raises(Exception, match="workspace smaller"):
        check(lib().amt_hpsi(plan.handle, prec, psi.data_ptr(), bare.data_ptr(), 7, 0, 3, v.data_ptr(),
                             ws.data_ptr(), 16, stream), "hpsi")


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_launch_shapes_give_identical_results(si_pseudo, precision):
    """Every launch shape the autotuner may pick (plane kernel of 256 or 512 threads, stick
    kernels over the default or half the sticks per workgroup) gives bit-identical H.psi on
    the Si8 k-batch (42^3); the hook rejects other shapes."""
    import torch

    from amaterasu_amd import ops
    from amaterasu_amd._lib import AmtError, check, lib
    from amaterasu_amd.device import DevicePlan
    from amaterasu_amd.system import build_system, load_dataset
    from amaterasu_amd.workloads import seeded_coefficients, si8_kbatch, smooth_potential

    spec = si8_kbatch(nk=3, nbands=9)
    s = build_system(spec.cell, spec.positions, spec.symbols, {"Si": load_dataset()}, spec.ecut_rho, spec.kpoints,
                     spec.ecuts)
    plan = DevicePlan(s.grid.shape, s.wave_spheres, s.projectors)
    prec = 1 if precision == "fp64" else 0
    cdt = torch.complex128 if prec else torch.complex64
    psi = torch.zeros((3, 9, plan.npw_pad), dtype=cdt, device="cuda")
    for k, sp in enumerate(s.wave_spheres):
        psi[k, :, : len(sp.g2)] = torch.from_numpy(seeded_coefficients(sp.g2, 9, seed=60 + k)).to("cuda", cdt)
    v = torch.from_numpy(smooth_potential(s.grid.shape, seed=6)).to("cuda", ops.real_dtype(prec))
    st = plan.sticks(prec, 27)
    wdef = 32 if prec else 64
    outs = []
    for nth in (256, 512):
        for w in (wdef, wdef // 2):
            check(lib().amt_plan_set_launch(plan.handle, prec, nth, w), "plan_set_launch")
            out = torch.zeros_like(psi)
            check(lib().amt_hpsi_local(plan.handle, prec, psi.data_ptr(), out.data_ptr(), 9, 0, 3, v.data_ptr(),
                                       st.data_ptr(), ops.stream_handle()), "hpsi_local")
            outs.append(out)
    torch.cuda.synchronize()
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    with pytest.raises(AmtError, match="plane_threads must be"):
        check(lib().amt_plan_set_launch(plan.handle, prec, 384, 0), "plan_set_launch")


@pytest.mark.parametrize("shape", [(21, 21, 21), (24, 24, 24), (45, 45, 45), (60, 60, 60), (63, 63, 63), (72, 72, 72),
                                   (84, 84, 84), (100, 100, 100), (108, 108, 108), (128, 128, 128),
                                   (24, 33, 33), (33, 24, 33), (33, 33, 24), (84, 20, 84), (20, 84, 84), (27, 108, 108)])
def test_plane_kernels_match_full_grid_route(shape):
    """Every plane kernel (one and four lanes per row, four-step) and every order of a grid with two
    equal axes, against the library's full-grid route on the same plan: H.psi and density of two
    ragged k-points, for spheres of the usual half width of the grid and for wide ones that reach
    past it (which the one-lane kernel leaves to the others). Bounds: a transform pair over N
    points is off by about log2(N) unit roundoffs of the largest value; 64 of them are allowed."""
    import torch

    from amaterasu_amd._lib import FP32, FP64
    from amaterasu_amd.basis import GSphere
    from amaterasu_amd.device import DevicePlan

    cell = np.diag(np.array(shape) / 4.0)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    n = min(shape)
    for half in (n / 4.0 - 0.4, min(n / 4.0 + 3.0, n / 2.0 - 2.0)):
        ecut = 0.5 * (half * 2.0 * np.pi / (n / 4.0)) ** 2
        spheres = [GSphere.build(cell, ecut * f, kpoint=np.array(k)) for f, k in ((1.0, (0, 0, 0)), (0.9, (0.4, -0.3, 0.1)))]
        nb = 3
        for prec, dt, u in ((FP32, torch.complex64, 2.0**-24), (FP64, torch.complex128, 2.0**-53)):
            plan = DevicePlan(shape, spheres)
            psi = torch.randn((2, nb, plan.npw_pad), dtype=dt, device="cuda", generator=g)
            for k in range(2):
                psi[k, :, plan.npw[k]:] = 0
            v = torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
            rows, weights = np.array([0, 2, 3, 5]), np.array([1.0, 0.5, 2.0, 0.25])
            got, rho = plan.hpsi(psi, v), torch.ones(shape, dtype=torch.float64, device="cuda")
            plan.accumulate_density(psi, rows, weights, rho, beta=0.5, scale=0.1, chunk=3)
            plan.set_route(prec, True)
            want, rho_want = plan.hpsi(psi, v), torch.ones(shape, dtype=torch.float64, device="cuda")
            plan.accumulate_density(psi, rows, weights, rho_want, beta=0.5, scale=0.1, chunk=3)
            bound = 64 * u * np.log2(np.prod(shape))
            assert float((got - want).abs().max() / want.abs().max()) < bound, (half, prec)
            assert float((rho - rho_want).abs().max() / rho_want.abs().max()) < bound, (half, prec)


@pytest.mark.parametrize("route", ["plane", "full grid"])
@pytest.mark.parametrize("split", [1, 7])
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("blocks", [[1], [8, 8, 8, 8], [1, 5, 18, 40, 130, 7], [31, 33, 97]])
def test_projector_contraction_and_padding(si2_system, blocks, dtype, split, route):
    """amt_hpsi with projector tables of any block lengths, with the first product split along the
    plane waves (splits summed and contracted in one launch) and not, against the local part plus
    the dense (psi beta^H) D beta in FP64: within the rounding of sums of npw, block and nproj
    terms. The output starts as NaN, so every element, padding included, has to be written."""
    import torch

    from amaterasu_amd import ops
    from amaterasu_amd._lib import check, lib
    from amaterasu_amd.hamiltonian import Hamiltonian

    dt = getattr(torch, dtype)
    rng = np.random.default_rng(len(blocks))
    v = rng.normal(size=(1, *si2_system.grid.shape))
    ham = Hamiltonian(si2_system, v, precision="fp64" if dtype == "complex128" else "fp32")
    plan = ham.plan
    plan.set_projectors(None)
    prec, nk, nb, np_, npw = ops.precision_of(torch.empty(0, dtype=dt)), plan.nk, 5, sum(blocks), plan.npw_pad
    rdt = ops.real_dtype(prec)
    live = torch.zeros(nk, 1, npw, dtype=torch.float64, device="cuda")
    for k in range(nk):
        live[k, :, : plan.npw[k]] = 1.0
    rand = lambda *s: torch.randn(*s, dtype=torch.complex128, device="cuda")  # noqa: E731
    torch.manual_seed(3)
    psi, beta = (rand(nk, nb, npw) * live).to(dt), (rand(nk, np_, npw) * live).to(dt)
    dij = torch.zeros(nk, np_, np_, dtype=rdt, device="cuda")
    starts = np.concatenate([[0], np.cumsum(blocks)])
    for a, n in zip(starts, blocks):
        d = torch.randn(nk, n, n, device="cuda", dtype=rdt)
        dij[:, a : a + n, a : a + n] = d + d.transpose(1, 2)
    start = torch.as_tensor(np.repeat(starts[:-1], blocks).astype(np.int32), device="cuda")
    length = torch.as_tensor(np.repeat(blocks, blocks).astype(np.int32), device="cuda")
    if route == "full grid":
        plan.set_route(prec, True)
    try:
        veff = ham.veff(0, prec)
        local = plan.hpsi(psi, veff)
        check(lib().amt_plan_set_projectors(plan.handle, prec, np_, beta.data_ptr(), dij.data_ptr(), start.data_ptr(),
                                            length.data_ptr()), "set_projectors")
        check(lib().amt_zgemm_set_split(prec, 1, nb, np_, npw, nk, split), "set_split")
        out = torch.full_like(psi, float("nan"))
        nbytes = lib().amt_hpsi_workspace(plan.handle, prec, nb, nk)
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        check(lib().amt_hpsi(plan.handle, prec, psi.data_ptr(), out.data_ptr(), nb, 0, nk, veff.data_ptr(), ws.data_ptr(),
                             nbytes, ops.stream_handle()), "hpsi")
    finally:
        lib().amt_zgemm_set_split(prec, 1, nb, np_, npw, nk, 0)
        lib().amt_plan_set_projectors(plan.handle, prec, 0, None, None, None, None)
        if route == "full grid":
            plan.set_route(prec, False)
    cpu = lambda t: t.cpu().to(torch.complex128)  # noqa: E731
    p64, b64, d64 = cpu(psi), cpu(beta), cpu(dij)
    want = cpu(local)
    size = want.abs()
    for k in range(nk):
        want[k] += (p64[k] @ b64[k].conj().T.contiguous()) @ d64[k] @ b64[k]
        size[k] += (p64[k].abs() @ b64[k].abs().T.contiguous()) @ d64[k].abs() @ b64[k].abs()
    u = 2.0**-53 if dtype == "complex128" else 2.0**-24
    # sums of length n err by at most about sqrt(n) u of the sum of absolute values here (random signs), 4 for the parts
    assert ((cpu(out) - want).abs() <= 4 * np.sqrt(npw + max(blocks) + np_) * u * size + 1e-300).all()
    assert not out[live.expand(nk, nb, npw) == 0].any() and out.isfinite().all()


@pytest.mark.parametrize("n,prec,one_lane", [(24, 0, True), (24, 1, True), (42, 0, True), (108, 1, True), (63, 0, False),
                                             (72, 0, False), (84, 1, False)])
def test_launch_tuning_by_plane_kernel(monkeypatch, n, prec, one_lane):
    """A narrow plan of a length with a one-lane plane kernel does not time plane workgroups, which
    that kernel has none to choose from; a wide plan of the same length has an entry of its own and
    is timed, whichever comes first."""
    import torch

    from amaterasu_amd import autotune
    from amaterasu_amd.basis import GSphere
    from amaterasu_amd.device import DevicePlan

    cell = np.eye(3) * n / 4.0
    monkeypatch.setenv("AMT_AUTOTUNE_FFT", "1")
    monkeypatch.setattr(autotune, "_FFT", {})
    stages = []
    timed = autotune._time_stage

    def record(plan, p, stage, *args, **kwargs):
        stages.append(stage)
        return timed(plan, p, stage, *args, **kwargs)

    monkeypatch.setattr(autotune, "_time_stage", record)
    v = torch.randn((n, n, n), dtype=torch.float64, device="cuda")
    for half, lanes in ((n / 4.0 - 0.4, one_lane), (n / 4.0 + 3.0, False)):
        plan = DevicePlan((n, n, n), [GSphere.build(cell, 0.5 * (half * 2.0 * np.pi / (n / 4.0)) ** 2)])
        assert bool(plan.info[16 + prec]) == lanes
        if not plan.plane_ok[prec]:
            continue  # a wide FP64 plane past LDS takes whole grids and has no launch shape
        psi = torch.randn((1, 2, plan.npw_pad), dtype=torch.complex128 if prec else torch.complex64, device="cuda")
        known = (n, prec, lanes) in autotune._FFT
        stages.clear()
        plan.hpsi(psi, v)
        assert (1 in stages) == (not known) and (2 in stages) == (not known and not lanes)
        stages.clear()
        plan.hpsi(psi, v)
        assert not stages and -1 not in (plan.info[12 + prec], plan.info[14 + prec])
    lanes_seen = {key[2] for key in autotune._FFT}
    assert lanes_seen == ({True, False} if one_lane and n <= 100 else {one_lane})
    for key, (nth, width) in autotune._FFT.items():
        assert (nth == 0) == key[2] and width in (16, 32, 64)


@pytest.mark.parametrize("shape", [(24, 20, 20), (20, 20, 24), (24, 24, 24)])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_first_call_of_a_length_under_capture(monkeypatch, shape, precision):
    """H.psi captured into a graph before its launch shapes are known: nothing is timed (that would
    wait for events inside the capture), and every replay, with eager calls and synchronisations in
    between, gives the eager result."""
    import torch

    from amaterasu_amd import autotune
    from amaterasu_amd.basis import GSphere
    from amaterasu_amd.device import DevicePlan

    n = min(shape)
    cell = np.diag(np.array(shape) / 4.0)
    dt = torch.complex64 if precision == "fp32" else torch.complex128
    plan = DevicePlan(shape, [GSphere.build(cell, 0.5 * ((n / 4.0 - 0.4) * 2.0 * np.pi / (n / 4.0)) ** 2)])
    g = torch.Generator(device="cuda").manual_seed(n)
    psi = torch.randn((1, 3, plan.npw_pad), dtype=dt, device="cuda", generator=g)
    v = torch.randn(shape, dtype=torch.float64 if precision == "fp64" else torch.float32, device="cuda", generator=g)
    monkeypatch.setattr(autotune, "_FFT", {})
    monkeypatch.setenv("AMT_AUTOTUNE_FFT", "0")
    out = torch.empty_like(psi)
    want = plan.hpsi(psi, v, out=out).clone()  # sizes the workspace
    monkeypatch.setenv("AMT_AUTOTUNE_FFT", "1")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.hpsi(psi, v, out=out)
    assert not autotune._FFT
    for _ in range(4):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(plan.hpsi(psi, v), want)
    assert len(autotune._FFT) == 1


def test_operator_workspace_holds_sticks_only():
    """An FP64 plane past LDS whose H.psi has the kernel with four lanes per row (108^2): amt_hpsi
    asks for the sticks of its rows and not for whole grids, which only the density takes there, and
    stays inside what it asked for."""
    import torch

    from amaterasu_amd import ops
    from amaterasu_amd._lib import FP64, check, lib
    from amaterasu_amd.basis import GSphere
    from amaterasu_amd.device import DevicePlan

    n, nb = 108, 3
    ecut = 0.5 * ((n / 4.0 - 0.4) * 2.0 * np.pi / (n / 4.0)) ** 2
    plan = DevicePlan((n, n, n), [GSphere.build(np.eye(3) * n / 4.0, ecut)])
    sticks = nb * n * plan.smax * 16
    nbytes = lib().amt_hpsi_workspace(plan.handle, FP64, nb, 1)
    assert sticks <= nbytes < sticks + 256
    assert lib().amt_plan_stick_bytes(plan.handle, FP64, nb) == nb * n**3 * 16
    g = torch.Generator(device="cuda").manual_seed(5)
    psi = torch.randn((1, nb, plan.npw_pad), dtype=torch.complex128, device="cuda", generator=g)
    v = torch.randn((n, n, n), dtype=torch.float64, device="cuda", generator=g)
    want = plan.hpsi(psi, v)
    ws = torch.full((nbytes + 4096,), 90, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(psi)
    check(lib().amt_hpsi(plan.handle, FP64, psi.data_ptr(), out.data_ptr(), nb, 0, 1, v.data_ptr(), ws.data_ptr(), nbytes,
                         ops.stream_handle()), "hpsi")
    torch.cuda.synchronize()
    assert torch.equal(out, want) and bool((ws[nbytes:] == 90).all())
    plan.set_route(FP64, True)
    assert lib().amt_hpsi_workspace(plan.handle, FP64, nb, 1) >= nb * n**3 * 16


LENGTHS = [20, 21, 22, 24, 25, 27, 28, 30, 32, 33, 35, 36, 40, 42, 44, 45, 48, 49, 50, 54, 55, 56, 60, 63, 64, 66, 70, 72,
           75, 77, 80, 81, 84, 88, 90, 96, 98, 99, 100, 105, 108, 110, 112, 120, 121, 126, 128]


@pytest.mark.parametrize("n", LENGTHS)
def test_plane_kernels_of_every_length(monkeypatch, n):
    """Every compile-time length against the library's full-grid route at a shifted k-point: on a
    sphere of the usual half width the one-lane kernel where the length has one, and on a wide one
    (and where it has none) the four-step kernel in both its workgroups, whose results are equal bits.
    Bound as for the orders of axes above: 64 log2(N) unit roundoffs of the largest value."""
    import torch

    from amaterasu_amd._lib import FP32, FP64, check, lib
    from amaterasu_amd.basis import GSphere
    from amaterasu_amd.device import DevicePlan

    monkeypatch.setenv("AMT_AUTOTUNE_FFT", "0")
    shape, nb = (n, n, n), 3
    g = torch.Generator(device="cuda").manual_seed(n)
    v = torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
    for half, wide in ((n / 4.0 - 0.4, False), (min(n / 4.0 + 3.0, n / 2.0 - 2.0), True)):
        sphere = GSphere.build(np.eye(3) * n / 4.0, 0.5 * (half * 2.0 * np.pi / (n / 4.0)) ** 2,
                               kpoint=np.array((0.4, -0.3, 0.1)))
        for prec, dt, u in ((FP32, torch.complex64, 2.0**-24), (FP64, torch.complex128, 2.0**-53)):
            plan = DevicePlan(shape, [sphere])
            lane, whole = plan.info[16 + prec], n * n * (16 if prec else 8) + 24 * n <= 160 * 1024
            assert not (wide and lane) and plan.plane_ok[prec] == bool(whole or lane)
            if not plan.plane_ok[prec]:
                continue
            psi = torch.randn((1, nb, plan.npw_pad), dtype=dt, device="cuda", generator=g)
            got = []
            for threads in (256, 512):
                check(lib().amt_plan_set_launch(plan.handle, prec, threads, 0), "plan_set_launch")
                got.append(plan.hpsi(psi, v))
            assert torch.equal(got[0], got[1])
            plan.set_route(prec, True)
            want = plan.hpsi(psi, v)
            err = float((got[0] - want).abs().max() / want.abs().max())
            assert err < 64 * u * np.log2(np.prod(shape)), (prec, wide)
