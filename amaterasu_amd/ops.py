"""Torch-level wrappers around the C ABI: tensors in, tensors out, on the current stream.

Every function here requires CUDA (HIP) tensors of the right dtype and layout and
raises otherwise; nothing falls back to a CPU implementation.
"""

from __future__ import annotations

import ctypes

import torch

from . import autotune
from ._lib import FP32, FP64, AmtError, check, lib

_WORKSPACES: dict = {}


def stream_handle() -> int:
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def precision_of(t: torch.Tensor) -> int:
    if t.dtype in (torch.complex128, torch.float64):
        return FP64
    if t.dtype in (torch.complex64, torch.float32):
        return FP32
    raise AmtError(f"unsupported dtype {t.dtype}")


def complex_dtype(prec: int):
    return torch.complex128 if prec == FP64 else torch.complex64


def real_dtype(prec: int):
    return torch.float64 if prec == FP64 else torch.float32


def _require(t: torch.Tensor, name: str):
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise AmtError(f"{name} must be a HIP device tensor")
    if not t.is_contiguous():
        raise AmtError(f"{name} must be contiguous")


def _require_rows(t: torch.Tensor, name: str):
    """A 2-D or 3-D device matrix (batch) whose rows are contiguous and do not overlap."""
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise AmtError(f"{name} must be a HIP device tensor")
    if t.dim() not in (2, 3):
        raise AmtError(f"{name} must be 2-D or 3-D")
    if t.shape[-1] > 1 and t.stride(-1) != 1:
        raise AmtError(f"{name} must have unit stride along its last axis")
    if t.shape[-2] > 1 and t.stride(-2) < t.shape[-1]:
        raise AmtError(f"{name} rows overlap")
    if t.dim() == 3 and t.shape[0] > 1 and t.stride(0) < t.shape[-2] * t.stride(-2) and t.shape[-2] > 0:
        raise AmtError(f"{name} batch entries overlap")


def workspace(nbytes: int, tag: str = "ws") -> torch.Tensor:
    """A cached device byte buffer of at least ``nbytes`` (grown, never shrunk)."""
    key = (tag, torch.cuda.current_device())
    buf = _WORKSPACES.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")
        _WORKSPACES[key] = buf
    return buf


def _scratch(nbytes: int) -> torch.Tensor:
    """A buffer of one call, from the current stream's pool: safe from several threads and streams
    (the allocation costs the host about 2 us)."""
    return torch.empty(int(nbytes), dtype=torch.uint8, device="cuda")


def zgemm(a: torch.Tensor, b: torch.Tensor, op: int, *, alpha: float = 1.0, beta: float = 0.0,
          out: torch.Tensor | None = None) -> torch.Tensor:
    """``alpha * a @ op(b) + beta * out`` on the matrix cores.

    ``op = 0``: b is (k, n). ``op = 1``: b is (n, k) and ``conj(b)^T`` is used.
    2-D operands, or 3-D operands batched over the leading axis.
    Operands may be strided views: each matrix needs unit stride along its rows' elements,
    a row stride of at least its column count and any batch stride.
    """
    _require_rows(a, "a")
    _require_rows(b, "b")
    if a.dtype != b.dtype or a.dtype not in (torch.complex64, torch.complex128):
        raise AmtError("zgemm operands must share a complex dtype")
    batched = a.dim() == 3
    a3 = a if batched else a.unsqueeze(0)
    b3 = b if batched else b.unsqueeze(0)
    nb, m, k = a3.shape
    if op == 0:
        kb, n = b3.shape[1], b3.shape[2]
    else:
        n, kb = b3.shape[1], b3.shape[2]
    if kb != k or b3.shape[0] != nb:
        raise AmtError(f"zgemm shape mismatch: a {tuple(a.shape)}, b {tuple(b.shape)}, op {op}")
    if out is None:
        if beta != 0.0:
            raise AmtError("beta != 0 needs out")
        out = torch.empty((nb, m, n) if batched else (m, n), dtype=a.dtype, device=a.device)
    _require_rows(out, "out")
    c3 = out if batched else out.unsqueeze(0)
    if tuple(c3.shape) != (nb, m, n):
        raise AmtError(f"zgemm out has shape {tuple(out.shape)}, expected {(nb, m, n)}")
    prec = precision_of(a)

    def launch(dst, al, be):
        wsb = lib().amt_zgemm_workspace(prec, op, m, n, k, nb)
        ws = workspace(wsb, "gemm") if wsb else None
        check(lib().amt_zgemm(prec, op, m, n, k, float(al), a3.data_ptr(), a3.stride(1), a3.stride(0),
                              b3.data_ptr(), b3.stride(1), b3.stride(0), float(be), dst.data_ptr(), dst.stride(1),
                              dst.stride(0), nb, ws.data_ptr() if ws is not None else None, int(wsb),
                              stream_handle()), "zgemm")

    if autotune.enabled() and autotune.bucket(prec, op, m, n, k, nb) not in autotune._TUNED:
        scratch = torch.empty((nb, m, n), dtype=a.dtype, device=a.device)
        autotune.tune_zgemm(lambda: launch(scratch, 1.0, 0.0), prec, op, m, n, k, nb)
        del scratch
    launch(c3, alpha, beta)
    return out


class _FFTPlan:
    """amt_fft_plan_create / amt_fft_plan_destroy for one grid shape on one device."""

    def __init__(self, shape):
        handle = ctypes.c_void_p()
        check(lib().amt_fft_plan_create(ctypes.byref(handle), *(int(n) for n in shape)), "fft_plan_create")
        self.handle = handle

    def __del__(self):
        h = getattr(self, "handle", None)
        if h is not None and h.value:
            try:
                lib().amt_fft_plan_destroy(h)
            except Exception:
                pass
            self.handle = None


_FFT_PLANS: dict = {}


def fft_plan(shape) -> "_FFTPlan":
    """The (cached) transform plan of a grid shape on the current device: its twiddle tables are
    allocated once here, so the transforms themselves allocate nothing."""
    key = (tuple(int(n) for n in shape), torch.cuda.current_device())
    plan = _FFT_PLANS.get(key)
    if plan is None:
        plan = _FFTPlan(key[0])
        _FFT_PLANS[key] = plan
    return plan


def fft3d(x: torch.Tensor, sign: int, scale: float = 1.0, *, inplace: bool = False) -> torch.Tensor:
    """Batched 3D transform over the last three axes (sign +1: e^{+iGr}, -1: e^{-iGr})."""
    _require(x, "x")
    y = x if inplace else x.clone()
    n1, n2, n3 = y.shape[-3:]
    batch = int(y.numel() // (n1 * n2 * n3))
    plan = fft_plan((n1, n2, n3))
    check(lib().amt_fft3d(plan.handle, precision_of(y), batch, y.data_ptr(), int(sign), float(scale),
                          stream_handle()), "fft3d")
    return y


def residual(hv: torch.Tensor, v: torch.Tensor, eps: torch.Tensor):
    """R = HV - eps V and ||R|| per row (float64)."""
    _require(hv, "hv")
    _require(v, "v")
    if hv.shape != v.shape or hv.dtype != v.dtype or v.dim() != 2:
        raise AmtError(f"residual: hv {tuple(hv.shape)} and v {tuple(v.shape)} must be equal 2-D blocks")
    nrow, npw = v.shape
    if eps.numel() != nrow:
        raise AmtError("residual: one eigenvalue per row")
    res = torch.empty_like(v)
    norms = torch.empty(nrow, dtype=torch.float64, device=v.device)
    e = eps.to(device=v.device, dtype=torch.float64).contiguous()
    check(lib().amt_residual(precision_of(v), hv.data_ptr(), v.data_ptr(), e.data_ptr(), res.data_ptr(),
                             norms.data_ptr(), nrow, npw, stream_handle()), "residual")
    return res, norms


def precondition(res: torch.Tensor, v: torch.Tensor, kinetic: torch.Tensor, rows: torch.Tensor, *,
                 rows_checked: bool = False) -> torch.Tensor:
    """Teter-Payne-Allan preconditioned, normalised residuals of the listed rows.
    ``rows_checked=True`` skips the range check of ``rows`` (two device reads), for callers
    whose rows come from indices of ``v`` itself (``nonzero`` of a per-row mask)."""
    _require(res, "res")
    _require(v, "v")
    if res.shape != v.shape or res.dtype != v.dtype or v.dim() != 2:
        raise AmtError("precondition: res and v must be equal 2-D blocks")
    prec = precision_of(v)
    kin = kinetic.to(device=v.device, dtype=torch.float64 if prec == FP64 else torch.float32).contiguous()
    if kin.numel() != v.shape[1]:
        raise AmtError("precondition: kinetic must have one entry per plane wave")
    r = rows.to(device=v.device, dtype=torch.int32).contiguous()
    if r.numel() and not rows_checked:
        lo, hi = torch.stack(torch.aminmax(r)).tolist()  # one device read
        if lo < 0 or hi >= v.shape[0]:
            raise AmtError("precondition: row index out of range")
    nout = int(r.numel())
    out = torch.empty((nout, v.shape[1]), dtype=v.dtype, device=v.device)
    check(lib().amt_precondition(prec, res.data_ptr(), v.data_ptr(), kin.data_ptr(), r.data_ptr(),
                                 out.data_ptr(), nout, v.shape[1], stream_handle()), "precondition")
    return out


def precondition_batched(res: torch.Tensor, v: torch.Tensor, kinetic: torch.Tensor, rows: torch.Tensor) -> torch.Tensor:
    """:func:`precondition` for all k-points in one launch: ``kinetic`` is ``[nk][npw]``, ``rows``
    ``[nk][width]`` (int32, device) holds row indices of ``res`` and ``v``, negative for a row of
    zeros, checked by the caller. Returns ``[nk][width][npw]``."""
    _require(res, "res")
    _require(v, "v")
    _require(kinetic, "kinetic")
    _require(rows, "rows")
    prec = precision_of(v)
    if res.shape != v.shape or res.dtype != v.dtype or v.dim() != 2:
        raise AmtError("precondition: res and v must be equal 2-D blocks")
    nk, width = rows.shape
    if rows.dtype != torch.int32 or kinetic.dtype != real_dtype(prec) or tuple(kinetic.shape) != (nk, v.shape[1]):
        raise AmtError("precondition: kinetic must have one entry per k-point and plane wave, rows one list per k-point")
    out = torch.empty((nk, width, v.shape[1]), dtype=v.dtype, device=v.device)
    check(lib().amt_precondition_batched(prec, res.data_ptr(), v.data_ptr(), kinetic.data_ptr(), rows.data_ptr(),
                                         out.data_ptr(), nk, width, v.shape[1], stream_handle()), "precondition_batched")
    return out


def append_rows(fresh: torch.Tensor, hfresh: torch.Tensor, basis: torch.Tensor, hbasis: torch.Tensor,
                grown: torch.Tensor):
    """Rows ``j < grown[1, k]`` of ``fresh`` and ``hfresh`` ``[nk][width][npw]`` become rows
    ``grown[0, k] + j`` of ``basis`` and ``hbasis`` ``[nk][cap][npw]`` (``grown`` int32, device)."""
    for t, name in ((fresh, "fresh"), (hfresh, "hfresh"), (basis, "basis"), (hbasis, "hbasis"), (grown, "grown")):
        _require(t, name)
    nk, width, npw = fresh.shape
    cap = basis.shape[1]
    if (hfresh.shape != fresh.shape or hbasis.shape != basis.shape or tuple(basis.shape) != (nk, cap, npw)
            or not fresh.dtype == hfresh.dtype == basis.dtype == hbasis.dtype):
        raise AmtError("append_rows: blocks of one dtype, [nk][width][npw] into [nk][cap][npw]")
    if grown.dtype != torch.int32 or tuple(grown.shape) != (2, nk):
        raise AmtError("append_rows: grown must be int32 [2][nk]")
    check(lib().amt_append_rows(precision_of(fresh), fresh.data_ptr(), hfresh.data_ptr(), basis.data_ptr(),
                                hbasis.data_ptr(), grown[0].data_ptr(), grown[1].data_ptr(), nk, width, cap, npw,
                                stream_handle()), "append_rows")


def append_projected(cols: torch.Tensor, proj: torch.Tensor, grown: torch.Tensor):
    """New rows and columns of the projected matrices ``proj`` ``[nk][cap][cap]`` from ``cols``
    ``[nk][cur][width]`` = basis (H fresh)^H; ``grown`` as in :func:`append_rows`."""
    for t, name in ((cols, "cols"), (proj, "proj"), (grown, "grown")):
        _require(t, name)
    nk, cur, width = cols.shape
    cap = proj.shape[1]
    if proj.dtype != torch.complex128 or tuple(proj.shape) != (nk, cap, cap) or cur > cap:
        raise AmtError("append_projected: proj must be complex128 [nk][cap][cap]")
    if grown.dtype != torch.int32 or tuple(grown.shape) != (2, nk):
        raise AmtError("append_projected: grown must be int32 [2][nk]")
    check(lib().amt_append_projected(precision_of(cols), cols.data_ptr(), proj.data_ptr(), grown[0].data_ptr(),
                                     grown[1].data_ptr(), nk, cur, width, cap, stream_handle()), "append_projected")


#: Gram matrices of at most this many rows go to the library's Cholesky and Loewdin kernels.
CHOL_MAX = 512


def _require_gram(gram: torch.Tensor):
    _require(gram, "gram")
    if gram.dtype not in (torch.complex64, torch.complex128) or gram.shape[-1] != gram.shape[-2]:
        raise AmtError("gram must be square complex matrices")
    if not 1 <= gram.shape[-1] <= CHOL_MAX:
        raise AmtError(f"gram has {gram.shape[-1]} rows, outside 1..{CHOL_MAX}")


def chol_inverse(gram: torch.Tensor, used: torch.Tensor | None = None):
    """(L^{-1}, stats) of the Hermitian part L L^H of a raw product block block^H, or of a batch of
    them with ``used`` (int32, device) leading rows each. See amt_chol_inverse: stats[..., 0] the
    status, [..., 1] the trace, [..., 2:] sums of |L^{-1}|^2."""
    _require_gram(gram)
    n, batch = gram.shape[-1], gram.numel() // gram.shape[-1] ** 2
    if used is not None and (used.dtype != torch.int32 or not used.is_cuda or used.numel() != batch):
        raise AmtError("used must be one int32 per matrix on the device")
    linv = torch.empty_like(gram)
    stats = torch.empty((*gram.shape[:-2], (n + 31) // 32 + 2), dtype=torch.float64, device=gram.device)
    nbytes = int(lib().amt_chol_workspace(n, batch))
    ws = _scratch(nbytes)
    check(lib().amt_chol_inverse(precision_of(gram), n, gram.data_ptr(), None if used is None else used.data_ptr(),
                                 batch, linv.data_ptr(), stats.data_ptr(), ws.data_ptr(), nbytes, stream_handle()),
          "chol_inverse")
    return linv, stats


def lowdin(gram: torch.Tensor):
    """(I - E/2 + 3 E^2/8, largest |component| of E per 32 rows), E = (gram + gram^H)/2 - I."""
    _require_gram(gram)
    n = gram.shape[-1]
    if gram.dim() != 2:
        raise AmtError("lowdin: one matrix")
    rot = torch.empty_like(gram)
    emax = torch.empty((n + 31) // 32, dtype=torch.float64, device=gram.device)
    check(lib().amt_lowdin(precision_of(gram), n, gram.data_ptr(), rot.data_ptr(), emax.data_ptr(), stream_handle()),
          "lowdin")
    return rot, emax


def heev_lowest(a: torch.Tensor, nev: int, *, workspace_tag: str | None = "heev"):
    """Lowest ``nev`` eigenpairs of a Hermitian complex128 matrix on the device: (w, zt) with
    w ascending (float64) and zt[k] the k-th eigenvector (row). See amt_heev_lowest. Calls
    that may run at the same time (on different streams) need different ``workspace_tag``s; ``None``
    takes scratch of this call."""
    _require(a, "a")
    if a.dtype != torch.complex128 or a.dim() != 2 or a.shape[0] != a.shape[1]:
        raise AmtError("heev: a must be a square complex128 device matrix")
    n = a.shape[0]
    if not 1 <= nev <= n:
        raise AmtError(f"heev: nev={nev} outside 1..{n}")
    w = torch.empty(nev, dtype=torch.float64, device=a.device)
    zt = torch.empty((nev, n), dtype=torch.complex128, device=a.device)
    nbytes = int(lib().amt_heev_workspace(n))
    ws = _scratch(nbytes) if workspace_tag is None else workspace(nbytes, workspace_tag)
    check(lib().amt_heev_lowest(n, a.data_ptr(), nev, w.data_ptr(), zt.data_ptr(), ws.data_ptr(), nbytes,
                                stream_handle()), "heev")
    return w, zt


def heev_lowest_batched(a: torch.Tensor, sizes, nev: int):
    """:func:`heev_lowest` of the leading ``sizes[k]`` rows of every matrix of ``a`` ``[nk][n][n]``
    (rows contiguous) in one set of launches: ``w`` ``[nk][nev]`` and ``zt`` ``[nk][nev][n]``, zero
    past ``sizes[k]``."""
    _require_rows(a, "a")
    if a.dtype != torch.complex128 or a.dim() != 3 or a.shape[1] != a.shape[2]:
        raise AmtError("heev: a must be square complex128 device matrices")
    nk, n = a.shape[0], a.shape[-1]
    sizes = [int(s) for s in sizes]
    if len(sizes) != nk or not all(1 <= nev <= s <= n for s in sizes):
        raise AmtError(f"heev: sizes {sizes} outside {nev}..{n}")
    w = torch.empty((nk, nev), dtype=torch.float64, device=a.device)
    zt = torch.empty((nk, nev, n), dtype=torch.complex128, device=a.device)
    nbytes = int(lib().amt_heev_batched_workspace(max(sizes), nk))
    ws = _scratch(nbytes)
    check(lib().amt_heev_lowest_batched(nk, (ctypes.c_int * nk)(*sizes), a.data_ptr(), a.stride(1), a.stride(0), nev,
                                        w.data_ptr(), zt.data_ptr(), n, ws.data_ptr(), nbytes, stream_handle()),
          "heev_batched")
    return w, zt



def finish_density(rho: torch.Tensor, volume: float = 1.0) -> torch.Tensor:
    """``rho / volume`` per spin, floored at zero and rescaled to the charge before the floor, in
    place (float64 ``[nspin][...]``); see amt_density_finish."""
    _require(rho, "rho")
    if rho.dtype != torch.float64 or rho.dim() < 2:
        raise AmtError("finish_density: rho must be float64 [nspin][...]")
    nspin = rho.shape[0]
    if rho.numel():
        part = _scratch(lib().amt_density_finish_bytes(nspin))
        check(lib().amt_density_finish(rho.data_ptr(), nspin, rho.numel() // nspin, float(volume), part.data_ptr(),
                                       stream_handle()), "density_finish")
    return rho


def gga(up, dn, suu, sud, sdd, parameters) -> torch.Tensor:
    """``[6][...]``: energy per particle, potentials and gradient derivatives of the PBE form at
    every point (float64); ``parameters`` = (kappa, mu, beta, gamma). See amt_gga."""
    fields = [f.contiguous() for f in (up, dn, suu, sud, sdd)]
    for f in fields:
        _require(f, "gga field")
        if f.dtype != torch.float64 or f.shape != fields[0].shape:
            raise AmtError("gga: float64 fields of one shape")
    out = torch.empty((6, *fields[0].shape), dtype=torch.float64, device=fields[0].device)
    n = fields[0].numel()
    if n:
        check(lib().amt_gga(n, *(f.data_ptr() for f in fields), (ctypes.c_double * 4)(*parameters), out.data_ptr(),
                            stream_handle()), "gga")
    return out
