"""Davidson on the GPU (scf/eigen/davidson.py:48-111) against dense LAPACK eigh and the
oracle, plus its fused residual and preconditioner kernels."""

from __future__ import annotations

import numpy as np
import pytest
from scipy.linalg import eigh

pytestmark = pytest.mark.gpu


def hermitian_operator(size=240, spread=40.0, coupling=0.02, seed=0):
    rng = np.random.default_rng(seed)
    d = np.sort(rng.uniform(0.0, spread, size))
    off = coupling * (rng.normal(size=(size, size)) + 1j * rng.normal(size=(size, size)))
    return np.diag(d) + off + off.conj().T, d


def test_dense_operator_matches_eigh():
    from amaterasu_amd.eigen import davidson, random_bands

    m, d = hermitian_operator()
    ref = eigh(m, eigvals_only=True)[:8]
    r = davidson(lambda b: b @ m.T, random_bands(len(d), 8, d, seed=1), d, tolerance=1e-10)
    assert r.converged
    assert np.abs(r.eigenvalues - ref).max() < 1e-11
    assert np.abs(r.coefficients @ r.coefficients.conj().T - np.eye(8)).max() < 1e-12


def test_residuals_bound_the_error():
    from amaterasu_amd.eigen import davidson, random_bands

    m, d = hermitian_operator(seed=4)
    ref = eigh(m, eigvals_only=True)[:5]
    r = davidson(lambda b: b @ m.T, random_bands(len(d), 5, d, seed=2), d, tolerance=1e-5, max_iterations=6)
    assert np.all(np.abs(r.eigenvalues - ref) <= r.residual_norms + 1e-14)


def test_random_bands_are_the_reference_draws():
    """Same default_rng stream as subspace.py:79-88: equal to the oracle up to the
    orthonormalisation's rounding."""
    from amaterasu_amd.eigen import random_bands
    from oracle.eigen import random_bands as orb

    t = np.linspace(0.0, 50.0, 300)
    a, b = random_bands(300, 6, t, seed=12345), orb(300, 6, t, seed=12345)
    assert np.abs(a - b).max() < 1e-12


def test_subspace_utilities():
    from amaterasu_amd.eigen import orthogonalize_against, orthonormalize, rayleigh_ritz

    rng = np.random.default_rng(0)
    b = orthonormalize(rng.normal(size=(5, 30)) + 1j * rng.normal(size=(5, 30)))
    assert np.abs(b @ b.conj().T - np.eye(5)).max() < 1e-12
    new = orthogonalize_against(rng.normal(size=(3, 30)) + 1j * rng.normal(size=(3, 30)), b)
    assert np.abs(new @ b.conj().T).max() < 1e-12
    assert np.abs(new @ new.conj().T - np.eye(len(new))).max() < 1e-12
    basis = orthonormalize(rng.normal(size=(4, 20)) + 0j)
    assert len(orthogonalize_against(basis[:2] + 1e-14 * rng.normal(size=(2, 20)), basis)) == 0
    m, _ = hermitian_operator(size=30, seed=9)
    q = orthonormalize(np.eye(30, dtype=complex))
    w, v, hv = rayleigh_ritz(q, q @ m.T, 30)
    assert np.abs(w - eigh(m, eigvals_only=True)).max() < 1e-12
    assert np.abs(hv - v @ m.T).max() < 1e-11


def test_residual_and_precondition_kernels():
    import torch

    from amaterasu_amd import ops
    from oracle.eigen import teter_payne_allan

    rng = np.random.default_rng(3)
    v = rng.normal(size=(7, 500)) + 1j * rng.normal(size=(7, 500))
    hv = rng.normal(size=(7, 500)) + 1j * rng.normal(size=(7, 500))
    eps = rng.normal(size=7)
    kin = np.linspace(0.0, 20.0, 500)
    res, norms = ops.residual(torch.from_numpy(hv).cuda(), torch.from_numpy(v).cuda(), torch.from_numpy(eps))
    ref = hv - eps[:, None] * v
    assert np.abs(res.cpu().numpy() - ref).max() < 1e-14
    assert np.abs(norms.cpu().numpy() - np.linalg.norm(ref, axis=1)).max() < 1e-12
    rows = np.array([0, 3, 6])
    out = ops.precondition(res, torch.from_numpy(v).cuda(), torch.from_numpy(kin), torch.from_numpy(rows))
    tb = np.einsum("ng,g->n", np.abs(v[rows]) ** 2, kin)
    c = teter_payne_allan(ref[rows], kin, tb)
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    assert np.abs(out.cpu().numpy() - c).max() < 1e-13


def test_davidson_with_gpu_hamiltonian_matches_oracle(si2_system):
    """The SCF's own call pattern (driver.py:345-353) on both paths from the same start."""
    from amaterasu_amd.eigen import solve
    from amaterasu_amd.hamiltonian import Hamiltonian
    from oracle.eigen import random_bands as orb
    from oracle.eigen import solve as osolve
    from oracle.hamiltonian import Hamiltonian as OH

    v = si2_system.v_local[None]
    h, o = Hamiltonian(si2_system, v), OH(si2_system, v)
    for ik, sp in enumerate(si2_system.wave_spheres):
        guess = orb(len(sp), 8, sp.kinetic_energy, seed=12345 + ik)
        a = solve("davidson", lambda b, ik=ik: h.apply(b, ik), guess, sp.kinetic_energy, tolerance=1e-9,
                  max_iterations=60)
        b = osolve("davidson", lambda x, ik=ik: o.apply(x, ik), guess, sp.kinetic_energy, tolerance=1e-9,
                   max_iterations=60)
        assert a.converged and b.converged
        assert np.abs(a.eigenvalues - b.eigenvalues).max() < 1e-10
        # same occupied subspace: projector difference
        pa, pb = a.coefficients[:4].T @ a.coefficients[:4].conj(), b.coefficients[:4].T @ b.coefficients[:4].conj()
        assert np.abs(pa - pb).max() < 1e-7


@pytest.mark.parametrize("dtype,cond_hard,orth", [("complex64", 1e3, 1e-5), ("complex128", 1e6, 1e-12)])
def test_orthonormalisation_refinement_and_its_fallback(monkeypatch, dtype, cond_hard, orth):
    """After the first Cholesky pass the rows of a well-conditioned block are orthonormal to
    within the Loewdin bound and take the refinement (no second factorisation); with the
    bound at zero the same block takes the second Cholesky pass; a block whose singular
    values spread over cond_hard goes whichever way its |E| sends it. Every result is
    orthonormal and spans the input rows."""
    import torch

    from amaterasu_amd import eigen

    calls = []
    second = eigen._cholesky_orthonormalize
    monkeypatch.setattr(eigen, "_cholesky_orthonormalize", lambda v: calls.append(1) or second(v))
    rng = np.random.default_rng(3)
    n, m = 4000, 24
    tdt = getattr(torch, dtype)

    def block_of(cond):
        u, _ = np.linalg.qr(rng.normal(size=(n, m)) + 1j * rng.normal(size=(n, m)))
        w, _ = np.linalg.qr(rng.normal(size=(m, m)) + 1j * rng.normal(size=(m, m)))
        return (w * np.geomspace(1.0, 1.0 / cond, m)) @ u.conj().T  # singular values 1 .. 1/cond

    def check(block, expect_calls):
        calls.clear()
        dev = torch.from_numpy(block).to(tdt).cuda()
        out = eigen._gram_orthonormalize(dev, 1e-7)
        if expect_calls is not None:
            assert len(calls) == expect_calls
        o = out.to(torch.complex128).cpu().numpy()
        b = dev.to(torch.complex128).cpu().numpy()
        assert o.shape == (m, n)
        assert np.abs(o @ o.conj().T - np.eye(m)).max() < orth
        assert np.abs((b @ o.conj().T) @ o - b).max() < (1e-3 if dtype == "complex64" else 1e-9)

    easy = block_of(2.0)
    check(easy, 0)
    monkeypatch.setitem(eigen._LOWDIN_MAX, tdt, 0.0)
    check(easy, 1)
    monkeypatch.undo()
    monkeypatch.setattr(eigen, "_cholesky_orthonormalize", lambda v: calls.append(1) or second(v))
    check(block_of(cond_hard), None)


@pytest.mark.parametrize("nb", [1, 2, 5, 20])
def test_small_projected_matrices(nb):
    """Projected matrices of 1 to 80 rows (the library's eigensolver from 2 on) in the per-k and the
    k-batched iteration, against the dense eigenvalues of the operator; an operator that is not
    finite raises, as zheevd did. Bound: residual norms below 1e-8 put an eigenvalue within 1e-8
    of the spectrum, and well within it by the gap (Weyl); 1e-8 is asserted."""
    import torch

    from amaterasu_amd.batched import solve_batched
    from amaterasu_amd.eigen import davidson

    n, nk = 300, 2
    g = torch.Generator(device="cuda").manual_seed(nb)
    kin = torch.linspace(0.1, 30.0, n, dtype=torch.float64, device="cuda").repeat(nk, 1)
    a = 0.05 * torch.randn((nk, n, n), dtype=torch.complex128, device="cuda", generator=g)
    a = (a + a.mH) / 2 + torch.diag_embed(kin.to(torch.complex128))
    guess = torch.randn((nk, nb, n), dtype=torch.complex128, device="cuda", generator=g) / (1 + kin[:, None, :])
    want = torch.stack([torch.linalg.eigvalsh(a[k].cpu()) for k in range(nk)])[:, :nb]
    each = [davidson(lambda x, k=k: x @ a[k].T.contiguous(), guess[k], kin[k], tolerance=1e-8, max_iterations=60)
            for k in range(nk)]
    both = solve_batched(lambda x: torch.stack([x[k] @ a[k].T.contiguous() for k in range(nk)]), guess, kin, [n] * nk,
                         tolerance=1e-8, max_iterations=60)
    for k in range(nk):
        assert each[k].converged and bool(both.converged[k])
        assert float((each[k].eigenvalues.cpu() - want[k]).abs().max()) < 1e-8
        assert float((both.eigenvalues[k].cpu() - want[k]).abs().max()) < 1e-8
    with pytest.raises(torch.linalg.LinAlgError):
        davidson(lambda x: x * float("nan"), guess[0], kin[0], tolerance=1e-8, max_iterations=3)
    with pytest.raises(torch.linalg.LinAlgError):
        solve_batched(lambda x: x * float("nan"), guess, kin, [n] * nk, tolerance=1e-8, max_iterations=3)


def _gram_with_spectrum(n, cond, rng):
    u, _ = np.linalg.qr(rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)))
    return (u * np.geomspace(1.0, 1.0 / cond, n)) @ u.conj().T


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 64, 65, 97, 160, 440, 512])
def test_inverse_cholesky_factor(dtype, n):
    """L^{-1} of a Gram matrix around the 32-row blocks: lower triangular, X G X^H = I within the
    factorisation's backward error (n u cond(G), eight of them; FP32 output adds its rounding of X,
    4 u32 cond(G) sqrt(n) in the Frobenius norm), the trace and the sums of |X|^2; a batch with
    fewer rows in use each (the rest the identity); the first pivot that is not positive."""
    import torch

    from amaterasu_amd import ops

    rng = np.random.default_rng(n)
    cond = 100.0
    u32 = 2.0**-24 if dtype == "complex64" else 0.0
    g = torch.from_numpy(_gram_with_spectrum(n, cond, rng)).to(getattr(torch, dtype))
    h = g.to(torch.complex128).numpy()
    h = 0.5 * (h + h.conj().T)
    bound = 8 * n * 2.0**-53 * cond + 4 * u32 * cond * np.sqrt(n)
    x, stats = ops.chol_inverse(g.cuda())
    x, stats = x.cpu().to(torch.complex128).numpy(), stats.cpu().numpy()
    assert stats[0] == 0 and np.abs(np.triu(x, 1)).max(initial=0.0) == 0.0
    assert np.linalg.norm(x @ h @ x.conj().T - np.eye(n)) <= bound
    assert abs(stats[1] - np.trace(h).real) <= n * 2.0**-53 * np.trace(h).real
    assert abs(stats[2:].sum() - np.sum(np.abs(x) ** 2)) <= (bound + 1e-14) * np.sum(np.abs(x) ** 2)
    used = [max(n // 2, 1), n, max(n - 1, 1)]
    batch = g.repeat(3, 1, 1).clone()
    for k, m in enumerate(used):
        batch[k, m:] = 0
        batch[k, :, m:] = 0
    x, stats = ops.chol_inverse(batch.cuda(), torch.tensor(used, dtype=torch.int32, device="cuda"))
    for k, m in enumerate(used):
        y = x[k].cpu().to(torch.complex128).numpy()
        assert float(stats[k, 0]) == 0
        assert np.linalg.norm(y[:m, :m] @ h[:m, :m] @ y[:m, :m].conj().T - np.eye(m)) <= bound
        assert np.array_equal(y[m:, m:], np.eye(n - m)) and not y[m:, :m].any()
        assert abs(float(stats[k, 2:].sum()) - np.sum(np.abs(y[:m, :m]) ** 2)) <= (bound + 1e-14) * np.sum(np.abs(y) ** 2)
    for bad in {0, n // 2, n - 1}:
        broken = g.clone()
        broken[bad, bad] = -1.0
        assert float(ops.chol_inverse(broken.cuda())[1][0]) == bad + 1
        broken[bad, bad] = float("nan")
        assert float(ops.chol_inverse(broken.cuda())[1][0]) == bad + 1
    # the Loewdin series of I + E
    e = 1e-3 * _gram_with_spectrum(n, 2.0, rng)
    v = torch.from_numpy(np.eye(n) + e).to(getattr(torch, dtype))
    e = v.to(torch.complex128).numpy()
    e = 0.5 * (e + e.conj().T) - np.eye(n)
    rot, emax = ops.lowdin(v.cuda())
    want = np.eye(n) - 0.5 * e + 0.375 * (e @ e)
    assert np.abs(rot.cpu().to(torch.complex128).numpy() - want).max() <= 2 * u32 + 4 * n * 2.0**-53
    assert float(emax.max()) == max(np.abs(e.real).max(), np.abs(e.imag).max())
    v[n // 2, 0] = float("nan")
    assert np.isnan(float(ops.lowdin(v.cuda())[1].cpu().max()))


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("last", [1, 2, 6])
def test_operator_that_stops_being_finite(bad, last):
    """One entry of H x that is not finite, in application ``last`` + 1 of ``last`` allowed iterations:
    the per-k and the k-batched iteration raise, also where no iteration is left to see it, and also
    when only one k-point is concerned; before, both return."""
    import torch

    from amaterasu_amd.batched import solve_batched
    from amaterasu_amd.eigen import davidson

    n, nb, nk = 200, 4, 2
    g = torch.Generator(device="cuda").manual_seed(last)
    kin = torch.linspace(0.1, 30.0, n, dtype=torch.float64, device="cuda").repeat(nk, 1)
    a = 0.2 * torch.randn((n, n), dtype=torch.complex128, device="cuda", generator=g)
    a = (a + a.mH) / 2 + torch.diag(kin[0].to(torch.complex128))
    guess = torch.randn((nk, nb, n), dtype=torch.complex128, device="cuda", generator=g) / (1 + kin[:, None, :])

    def operator(at):
        calls = []

        def apply(x):
            calls.append(1)
            out = x @ a.T.contiguous()
            if len(calls) == at:
                out[..., -1, 3] = bad
                if out.dim() == 3:
                    out[0] = x[0] @ a.T.contiguous()
            return out

        return apply

    for at, raises in ((last + 2, False), (last + 1, True), (1, True)):
        if raises:
            with pytest.raises(torch.linalg.LinAlgError):
                davidson(operator(at), guess[0], kin[0], tolerance=1e-10, max_iterations=last)
            with pytest.raises(torch.linalg.LinAlgError):
                solve_batched(operator(at), guess, kin, [n] * nk, tolerance=1e-10, max_iterations=last)
        else:
            one = davidson(operator(at), guess[0], kin[0], tolerance=1e-10, max_iterations=last)
            both = solve_batched(operator(at), guess, kin, [n] * nk, tolerance=1e-10, max_iterations=last)
            assert bool(torch.isfinite(one.eigenvalues).all()) and bool(torch.isfinite(both.eigenvalues).all())


def test_small_eigensolves_share_no_scratch(monkeypatch):
    """Projected matrices of 2 to 95 rows: no cached workspace is used, and solves on two threads,
    each on its own stream, give the bits of solves alone."""
    import threading

    import torch

    from amaterasu_amd import eigen, ops

    g = torch.Generator(device="cuda").manual_seed(0)
    mats = [torch.randn((n, n), dtype=torch.complex128, device="cuda", generator=g) for n in (2, 20, 80, 95)]
    mats = [a + a.mH for a in mats]
    alone = [eigen._lowest_eigenpairs(a, max(len(a) // 4, 1)) for a in mats]
    torch.cuda.synchronize()

    def refuse(*args):
        raise AssertionError("a cached workspace was asked for")

    monkeypatch.setattr(ops, "workspace", refuse)
    different, finished = [], []

    def work(order):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                got = [(i, eigen._lowest_eigenpairs(mats[i], max(len(mats[i]) // 4, 1))) for i in order]
                torch.cuda.current_stream().synchronize()
                different.extend(i for i, (w, z) in got
                                 if not (torch.equal(w, alone[i][0]) and torch.equal(z, alone[i][1])))
        finished.append(order)

    threads = [threading.Thread(target=work, args=(order,)) for order in ((0, 1, 2, 3), (3, 2, 1, 0))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(finished) == 2 and not different
