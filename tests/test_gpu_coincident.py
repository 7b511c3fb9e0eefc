"""Symmetric products with a coincidence shift on both sides of the pair split:
eight workgroups a tile pair (600 and 13000 points) and one (20481), with coincident
points in tiles of their own and in others."""
import ctypes as C

import numpy as np
import pytest

from mpla_amd import _native
from tests.gpu_util import host, require_gpu, stream, workspace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    require_gpu()
    return _native.mplak()


@pytest.mark.parametrize("n,dim", [(600, 1), (13000, 2), (20481, 3)])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("prec,bar", [(_native.MPLAK_PREC_F64, 1e-12), (_native.MPLAK_PREC_F32, 2e-5)])
def test_symmetric_products_with_coincident_points(lib, monkeypatch, n, dim, kind, prec, bar):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    P = P[:, torch.argsort(P[0])].contiguous()
    P[:, 9::100] = P[:, 8::100][:, :P[:, 9::100].shape[1]]  # neighbours
    P[:, n - 40:] = P[:, 100:500:10]                        # the last tile repeats points of the first one
    x = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
    ell, nugget, shift = (0.05, 0.1)[kind], 0.5, 0.25
    ref, mag = torch.empty_like(x), torch.empty_like(x)
    for i in range(0, n, 4096):
        s = sum((P[d, i:i + 4096, None] - P[d][None]) ** 2 for d in range(dim))
        r = (3.0 * s).sqrt() / ell
        K = ((-0.5 * s / ell ** 2).exp() if kind == 0 else (1.0 + r) * (-r).exp()) + shift * (s == 0)
        ref[i:i + 4096], mag[i:i + 4096] = K @ x, K @ x.abs()
    ref, mag = host(ref + nugget * x), host(mag + nugget * x.abs())
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, kind, ell, nugget, shift, 0, n, 0, n)
    monkeypatch.setenv("MPLAK_KMV_SYMMETRIC", "1")
    wb = lib.mplak_kernel_matvec_workspace_bytes(C.byref(desc))
    y = torch.empty_like(x)

    def product(form):
        y.fill_(7.0)
        if form == "planned":
            pb = lib.mplak_screen_plan_bytes(C.byref(desc))
            plan = workspace(pb)
            plan.fill_(float("nan"))
            _native.check(lib.mplak_screen_plan_build(C.byref(desc), prec, 2000.0, plan.data_ptr(), pb, stream()))
            _native.check(lib.mplak_kernel_matvec_planned(C.byref(desc), prec, 2000.0, plan.data_ptr(), pb,
                                                          x.data_ptr(), y.data_ptr(), None, stream()))
        else:
            w = workspace(wb)
            w.fill_(float("nan"))
            args = (x.data_ptr(), y.data_ptr(), w.data_ptr(), wb, None, stream())
            if form == "exact":
                _native.check(lib.mplak_kernel_matvec(C.byref(desc), prec, *args))
            else:
                _native.check(lib.mplak_kernel_matvec_screened(C.byref(desc), prec, 2000.0, *args))
        return host(y).copy()

    exact = product("exact")
    assert np.all(np.abs(exact - ref) <= bar * mag)
    for form in ("screened", "planned"):  # nothing is dropped
        assert np.array_equal(product(form), exact), form
