"""The MFMA complex GEMM (NN and NC, FP64 and FP32, split-K, batched) against numpy."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _c(shape, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(size=shape) + 1j * rng.normal(size=shape)


@pytest.mark.parametrize("dtype,tol", [("complex128", 1e-13), ("complex64", 2e-5)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (17, 33, 9), (64, 64, 16), (100, 70, 300), (8, 36, 754),
                                   (160, 1152, 3000), (37, 5, 40000), (300, 270, 1000), (257, 513, 700),
                                   (256, 384, 3000), (150, 90, 700), (470, 33, 5000), (150, 20000, 1100)])
def test_zgemm_nn_and_nc(dtype, tol, m, n, k):
    """Every tile shape: 64- and 128-row tiles, 80-row tiles with ragged edges (m = 150, 470),
    and an 80-row candidate whose single K chunk would need the two-level kernel (m = 150,
    k = 1100 with 626 output tiles: it falls back to 64-row tiles)."""
    import torch

    from amaterasu_amd import ops

    a, b_nn, b_nc = _c((m, k), 1), _c((k, n), 2), _c((n, k), 3)
    ta = torch.from_numpy(a).to("cuda", getattr(torch, dtype))
    nn = ops.zgemm(ta, torch.from_numpy(b_nn).to("cuda", ta.dtype), 0).cpu().numpy()
    nc = ops.zgemm(ta, torch.from_numpy(b_nc).to("cuda", ta.dtype), 1).cpu().numpy()
    ref_nn, ref_nc = a @ b_nn, a @ b_nc.conj().T
    scale = np.sqrt(k) * 2.0
    assert np.abs(nn - ref_nn).max() / scale < tol
    assert np.abs(nc - ref_nc).max() / scale < tol


def test_zgemm_alpha_beta_and_batch():
    import torch

    from amaterasu_amd import ops

    a, b, c = _c((3, 20, 50), 4), _c((3, 50, 30), 5), _c((3, 20, 30), 6)
    tc = torch.from_numpy(c).cuda()
    ops.zgemm(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), 0, alpha=-1.0, beta=1.0, out=tc)
    assert np.abs(tc.cpu().numpy() - (c - a @ b)).max() < 1e-12
    bc = _c((3, 30, 50), 7)
    out = ops.zgemm(torch.from_numpy(a).cuda(), torch.from_numpy(bc).cuda(), 1).cpu().numpy()
    assert np.abs(out - a @ bc.conj().transpose(0, 2, 1)).max() < 1e-12


def test_mfma_lane_layout_single_tile():
    """A 16x16x4 product with distinct small integers: exact in both precisions, so any
    lane-layout mistake (transposed fragment, wrong row of the accumulator) shows up as
    a wrong integer."""
    import torch

    from amaterasu_amd import ops

    a = (np.arange(16 * 4).reshape(16, 4) % 7 + 1j * (np.arange(64).reshape(16, 4) % 5)).astype(np.complex128)
    b = (np.arange(4 * 16).reshape(4, 16) % 3 - 1j * (np.arange(64).reshape(4, 16) % 4)).astype(np.complex128)
    for dt in (torch.complex128, torch.complex64):
        got = ops.zgemm(torch.from_numpy(a).to("cuda", dt), torch.from_numpy(b).to("cuda", dt), 0).cpu().numpy()
        assert np.array_equal(got.astype(np.complex128), a @ b)


def test_zgemm_strided_views():
    """Row-strided and batch-strided views (a prefix of a larger subspace block) go to the
    kernel without copies and give the same products."""
    import torch

    from amaterasu_amd import ops

    g = torch.Generator().manual_seed(5)
    big = torch.randn((3, 40, 130), dtype=torch.complex128, generator=g).cuda()
    a = torch.randn((3, 7, 130), dtype=torch.complex128, generator=g).cuda()
    view = big[:, :25]  # batch stride 40*130, rows of 130
    c = ops.zgemm(a, view, 1)
    want = a.cpu() @ view.cpu().conj().transpose(-1, -2)
    assert torch.allclose(c.cpu(), want, rtol=1e-12, atol=1e-11)
    rot = torch.randn((3, 5, 25), dtype=torch.complex128, generator=g).cuda()
    out = torch.zeros((3, 9, 130), dtype=torch.complex128).cuda()
    ops.zgemm(rot, view, 0, out=out[:, 2:7])
    assert torch.allclose(out[:, 2:7].cpu(), rot.cpu() @ view.cpu(), rtol=1e-12, atol=1e-11)
    assert float(out[:, :2].abs().max()) == 0.0 and float(out[:, 7:].abs().max()) == 0.0


@pytest.mark.parametrize("split", [1, 0])
def test_zgemm_fp32_long_contraction_accumulates_in_fp64(split):
    """Gram matrix of unit rows over K = 131072 plane waves in FP32 against the FP64 product
    of the same (FP32-rounded) inputs. With one split (the whole contraction in one
    workgroup) the FP32 matrix-core sums are carried into FP64 every 64 of K; with the
    heuristic split (256 chunks of 512) each chunk keeps one FP32 accumulator and the
    partials are summed in FP64. Either way the error stays near the final rounding
    (~1e-7), where one FP32 accumulator over all of K loses ~1e-4 on the unit diagonal."""
    import torch

    from amaterasu_amd import ops
    from amaterasu_amd._lib import FP32, check, lib

    m, k = 128, 131072
    g = torch.Generator().manual_seed(9)
    a = torch.randn((m, k), dtype=torch.complex128, generator=g)
    a = (a / torch.linalg.vector_norm(a, dim=1, keepdim=True)).to(torch.complex64).cuda()
    a64 = a.to(torch.complex128)
    check(lib().amt_zgemm_set_split(FP32, 1, m, m, k, 1, split), "zgemm_set_split")
    try:
        got = ops.zgemm(a, a, 1).to(torch.complex128)
    finally:
        check(lib().amt_zgemm_set_split(FP32, 1, m, m, k, 1, 0), "zgemm_set_split")
    want = ops.zgemm(a64, a64, 1)
    assert float((torch.diagonal(want) - 1.0).abs().max()) < 1e-6
    assert float((got - want).abs().max()) < 3e-7


def test_zgemm_fp32_large_tiles_long_contraction():
    """FP32 NC products with both output sides >= 256 take 128 x 128 tiles with K chunks of
    512 and the FP64 split reduction: the same K = 131 072 unit-row Gram check (batched, so
    the batch offsets of the partial products are exercised too), and an NN rotation of the
    same rows."""
    import torch

    from amaterasu_amd import ops

    nb, m, k = 2, 256, 131072
    g = torch.Generator().manual_seed(10)
    a = torch.randn((nb, m, k), dtype=torch.complex128, generator=g)
    a = (a / torch.linalg.vector_norm(a, dim=-1, keepdim=True)).to(torch.complex64).cuda()
    a64 = a.to(torch.complex128)
    got = ops.zgemm(a, a, 1).to(torch.complex128)
    want = ops.zgemm(a64, a64, 1)
    assert float((got - want).abs().max()) < 3e-7
    rot = torch.randn((nb, 300, m), dtype=torch.complex128, generator=g).cuda() / m**0.5
    got = ops.zgemm(rot.to(torch.complex64), a, 0).to(torch.complex128)
    want = ops.zgemm(rot.to(torch.complex64).to(torch.complex128), a64, 0)
    # single-level FP32 over K = 256 in Gauss's three-product form: the imaginary part's
    # rounding is bounded by eps * sum |a_re + a_im| |b_re + b_im|, up to twice the bound of
    # four real products (measured 1.1e-6 here; the four-product form passed 1e-6)
    assert float((got - want).abs().max() / want.abs().max()) < 2e-6


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("m", [1, 15, 17, 33, 48, 65, 80, 97, 112, 113, 160])
def test_zgemm_tile_edges(dtype, m):
    """Every tile height (16 to 112 rows) with one row more or less, against numpy in FP64 on the
    same inputs: columns around the 64 of a tile and the two of an FP32 chunk, K around one, two
    and four K tiles (8 or 16) and past the length that carries FP64 sums, row strides that leave
    rows 8-byte aligned. The bound is the summation's own: with u the unit roundoff, a sum of k
    products in one accumulator is off by at most (k + 8) u times the sum of the magnitudes, in the
    three-product form at most three times that (an FP32 accumulator covers at most 1024 of k). A
    NaN in the last row of A stays in the last row of the product."""
    import torch

    from amaterasu_amd import ops

    u = 2.0**-53 if dtype == "complex128" else 2.0**-24
    dt = getattr(torch, dtype)
    for n in (1, 2, 63, 64, 65, 131):
        for k in (1, 7, 8, 9, 16, 17, 33, 64, 127, 1027, 2051):
            big = torch.from_numpy(_c((m, k + 3), m + k)).to(dt)
            bnn, bnc = torch.from_numpy(_c((k, n + 1), n)).to(dt), torch.from_numpy(_c((n, k + 1), n + 7)).to(dt)
            a = big[:, 1 : 1 + k]
            for op, b in ((0, bnn[:, :n]), (1, bnc[:, :k])):
                dev = [x.cuda() for x in (big, bnn if op == 0 else bnc)]
                da, db = dev[0][:, 1 : 1 + k], dev[1][:, :n] if op == 0 else dev[1][:, :k]
                got = ops.zgemm(da, db, op).cpu().to(torch.complex128).numpy()
                x, y = a.to(torch.complex128).numpy(), b.to(torch.complex128).numpy()
                y = y if op == 0 else y.conj().T
                size = (np.abs(x.real) + np.abs(x.imag)) @ (np.abs(y.real) + np.abs(y.imag))
                assert (np.abs(got - x @ y) <= 3.0 * (min(k, 1024) + 8) * u * size).all(), (n, k, op)
        if m > 1:
            bad = dev[0].clone()
            bad[-1] = float("nan")
            got = ops.zgemm(bad[:, 1 : 1 + k], db, op)
            assert bool(torch.isfinite(torch.view_as_real(got[:-1])).all()) and bool(got[-1].isnan().all())


@pytest.mark.parametrize("op,m,n,k,batch", [(0, 80, 18500, 576, 1), (0, 58, 13900, 432, 1), (0, 40, 9301, 288, 1),
                                            (0, 17, 1830, 399, 5), (0, 5, 700, 1024, 1), (0, 9, 3000, 1500, 1),
                                            (1, 19, 1381, 355, 5), (1, 264, 19, 391, 3), (1, 300, 270, 461, 1),
                                            (1, 28, 3011, 6522, 11), (1, 64, 33000, 1100, 1), (1, 160, 480, 9000, 1)])
def test_zgemm_fp32_accumulator_length(op, m, n, k, batch):
    """K that one FP32 accumulator may cover: the equal parts of at most 256 that K divides into (to
    the next K tile of 16), 64 where an NC product has 512 tiles of 64 x 64 outputs and more than
    1024 of K. Integers whose sums are exact in FP32 up to that length and not beyond, so only two
    roundings are left: of each partial product and of the result, at most u times the (positive)
    sum each; an accumulator of twice the length loses several units in the last place."""
    import torch

    from amaterasu_amd import ops

    parts = (k + 255) // 256
    length = (-(-k // parts) + 15) // 16 * 16
    if op == 1 and k > 1024 and -(-m // 64) * -(-n // 64) * batch >= 512:
        length = 64
    top = 2**24 // length
    g = torch.Generator(device="cuda").manual_seed(k)
    b = torch.randint(top - top // 20, top + 1, (batch, k, n) if op == 0 else (batch, n, k), device="cuda", generator=g)
    want = b.sum(1 if op == 0 else 2)[:, None, :].to(torch.float64)
    a = torch.ones((batch, m, k), dtype=torch.complex64, device="cuda")
    got = ops.zgemm(a, b.to(torch.complex64), op)
    assert not got.imag.any()
    assert bool(((got.real.to(torch.float64) - want).abs() <= 2 * 2.0**-24 * want).all())


@pytest.mark.parametrize("op,m,n,k,batch", [(0, 80, 18500, 576, 1), (0, 58, 13900, 432, 1), (0, 80, 18500, 1000, 1),
                                            (0, 52, 5241, 272, 4), (0, 133, 7390, 288, 2), (0, 178, 8418, 621, 1),
                                            (1, 19, 1381, 355, 5), (1, 83, 7159, 265, 2), (1, 133, 7946, 303, 2),
                                            (1, 180, 3826, 1382, 1), (1, 40, 288, 9300, 4)])
def test_zgemm_fp64_accumulator_length(op, m, n, k, batch):
    """FP64 products of 257 and more of K sum it in pieces of at most 192, of 1 to 4 tile heights.
    Integers whose sums are exact up to that length: what is left is one rounding for each piece
    added, of half a unit of the (positive) sum at most, and no more than K / 64 + 1 of them; one
    accumulator over all of K rounds at every fourth of K past 192."""
    import torch

    from amaterasu_amd import ops

    top = 2**53 // 192
    g = torch.Generator(device="cuda").manual_seed(k)
    b = torch.randint(top - top // 20, top + 1, (batch, k, n) if op == 0 else (batch, n, k), device="cuda", generator=g)
    want = b.sum(1 if op == 0 else 2)[:, None, :]
    a = torch.ones((batch, m, k), dtype=torch.complex128, device="cuda")
    got = ops.zgemm(a, b.to(torch.complex128), op)
    assert not got.imag.any()
    bound = (k / 64 + 1) * 2.0**-53 * want.to(torch.float64)
    assert bool(((got.real.to(torch.int64) - want).abs().to(torch.float64) <= bound).all())
