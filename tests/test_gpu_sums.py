"""Accuracy of the products' sums over many sources or columns.

A running sum of k terms of random sign, rms sigma, has rms sqrt(k) sigma, and
each of its roundings is a uniform error of rms 0.425 u of the sum (u half the
spacing at 1; averaged over the logarithm of the mantissa).  A chain of L terms
therefore errs by 0.425 u sigma L / sqrt(2), n / L such chains by 0.425 u sigma
sqrt(n L / 2), and relative to the result, of rms sqrt(n) sigma, by 0.425 u
sqrt(L / 2) whatever n."""
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


def sum_error(lib, n, R, kind, prec, rows=64, cols=16):
    """Relative 2-norm error of the first rows and columns of K V, V of random sign."""
    import torch
    dim, ell = (3, 2)[kind], 0.3
    g = torch.Generator(device="cuda").manual_seed(n + R)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    V = torch.rand((R, n), generator=g, dtype=torch.float64, device="cuda") - 0.5
    Y = torch.empty_like(V)
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, kind, ell, 0.0, 0.0, 0, n, 0, n)
    wb = lib.mplak_kernel_mrhs_workspace_bytes(C.byref(desc), prec, R)
    w = workspace(wb)
    _native.check(lib.mplak_kernel_mrhs(C.byref(desc), prec, R, V.data_ptr(), n, Y.data_ptr(), n, w.data_ptr(), wb,
                                        None, stream()))
    got = host(Y)[:cols, :rows]
    Pl = host(P).astype(np.longdouble)
    s = sum((Pl[d, :rows, None] - Pl[d][None]) ** 2 for d in range(dim))
    r = np.sqrt(3 * s) / np.longdouble(ell)
    K = np.exp(-s / (2 * np.longdouble(ell) ** 2)) if kind == 0 else (1 + r) * np.exp(-r)
    ref = host(V)[:cols].astype(np.longdouble) @ K.T
    return float(np.sqrt(((got - ref) ** 2).sum() / (ref ** 2).sum()))


# FP64 on the matrix cores (one to four 16-column blocks): chains of 256 sources.
# With u for 0.425 u, and 8 u for the entries and the sums of chains and slabs.
@pytest.mark.parametrize("R", [16, 32, 48, 64])
@pytest.mark.parametrize("kind", [0, 1])
def test_mrhs_f64_sums_in_short_chains(lib, R, kind):
    assert sum_error(lib, 50000, R, kind, _native.MPLAK_PREC_F64) <= 2.0 ** -53 * (np.sqrt(256 / 2) + 8)


# FP32 on the matrix cores: chains of at most 512 sources at 16000 points (FP64
# sums of them); a quarter on top for the entries' few roundings.
@pytest.mark.parametrize("R", [32, 64])
@pytest.mark.parametrize("kind", [0, 1])
def test_mrhs_f32_sums_in_short_chains(lib, R, kind):
    bound = 1.25 * 0.425 * 2.0 ** -24 * np.sqrt(512 / 2)
    assert sum_error(lib, 16000, R, kind, _native.MPLAK_PREC_F32) <= bound


# Streamed dense products: running sums of 256 columns, added over a wave's
# thousands of columns (one slab and several; odd strides), then over the waves.
@pytest.mark.parametrize("m,n,lda", [(20000, 16000, 20000), (16385, 16385, 16387), (140000, 4001, 140000)])
def test_dgemv_sums_in_short_chains(lib, m, n, lda):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.rand((n, lda), generator=g, dtype=torch.float64, device="cuda") - 0.5
    x = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
    y = torch.empty(m, dtype=torch.float64, device="cuda")
    wb = lib.mplak_dgemv_workspace_bytes(m, n)
    w = workspace(wb)
    _native.check(lib.mplak_dgemv_f64(m, n, A.data_ptr(), lda, x.data_ptr(), y.data_ptr(), w.data_ptr(), wb, None,
                                      stream()))
    rows = slice(m // 2, m // 2 + 200)
    ref = host(A[:, rows]).T.astype(np.longdouble) @ host(x).astype(np.longdouble)
    error = float(np.sqrt(((host(y)[rows] - ref) ** 2).sum() / (ref ** 2).sum()))
    # chains of 256, up to n / 256 of them in a row, and the last sums
    assert error <= 0.425 * 2.0 ** -53 * (np.sqrt(256 / 2) + np.sqrt(n / 256 / 2) + 2)


# Planned FP32 Matern products form squared distances on the vector unit in 1-D
# and 2-D, on the matrix cores in 3-D: the same points with coordinates of zero
# added are as accurate either way.
@pytest.mark.parametrize("n", [2000, 4096, 8000])
@pytest.mark.parametrize("dim,ell", [(1, 0.02), (2, 0.1)])
def test_planned_fp32_distances_of_both_forms(lib, n, dim, ell):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    ob = lib.mplak_spatial_order_workspace_bytes(n, dim)
    w, perm = workspace(ob), torch.empty(n, dtype=torch.int64, device="cuda")
    _native.check(lib.mplak_spatial_order(table.data_ptr(), dim, 0, n, perm.data_ptr(), w.data_ptr(), ob, stream()))
    P = torch.cat([P[:, perm], torch.zeros((3 - dim, n), dtype=torch.float64, device="cuda")]).contiguous()
    x = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
    r = (3.0 * sum((P[d, :, None] - P[d][None]) ** 2 for d in range(dim))).sqrt() / ell
    ref = ((1.0 + r) * (-r).exp()) @ x + x
    table = torch.tensor([P[d].data_ptr() for d in range(3)], dtype=torch.int64, device="cuda")
    error = {}
    for form in (dim, 3):
        desc = _native.mplak_kernel_desc(table.data_ptr(), form, 1, ell, 1.0, 0.0, 0, n, 0, n)
        pb = lib.mplak_screen_plan_bytes(C.byref(desc))
        plan, y = workspace(pb), torch.empty_like(x)
        _native.check(lib.mplak_screen_plan_build(C.byref(desc), _native.MPLAK_PREC_F32, 40.0, plan.data_ptr(), pb,
                                                  stream()))
        _native.check(lib.mplak_kernel_matvec_planned(C.byref(desc), _native.MPLAK_PREC_F32, 40.0, plan.data_ptr(), pb,
                                                      x.data_ptr(), y.data_ptr(), None, stream()))
        error[form] = float((y - ref).norm() / ref.norm())
    assert error[dim] <= 1.05 * error[3]


# Few targets and many sources: many slabs, whose partials a finish workgroup adds
# in 2 to 256 slices (256 to 1 rows), and just too few slabs or too many rows for it.
@pytest.mark.parametrize("rows,cols,R", [(1, 20011, 1), (2, 3000, 64), (3, 70001, 16), (65, 20000, 9), (127, 2111, 5),
                                         (200, 65536, 64), (257, 30000, 8), (1000, 20000, 64), (1, 500, 3)])
@pytest.mark.parametrize("prec,bar", [(_native.MPLAK_PREC_F64, 1e-12), (_native.MPLAK_PREC_F32, 2e-5),
                                      (_native.MPLAK_PREC_BF16X3, 1e-4)])
def test_mrhs_few_targets(lib, rows, cols, R, prec, bar):
    import torch
    dim, ell, off, nugget, ldv, ldy = 3, 0.3, 5, 0.7, cols + 1, rows + 2
    g = torch.Generator(device="cuda").manual_seed(cols + R)
    P = torch.rand((dim, cols + off), generator=g, dtype=torch.float64, device="cuda")
    V = torch.randn((R, ldv), generator=g, dtype=torch.float64, device="cuda")
    Y = torch.full((R, ldy), 7.0, dtype=torch.float64, device="cuda")
    K = (-sum((P[d, off:off + rows, None] - P[d][None, :cols]) ** 2 for d in range(dim)) / (2 * ell ** 2)).exp()
    K[torch.arange(rows), torch.arange(rows) + off] += nugget
    ref, mag = host(V[:, :cols] @ K.t()), host(V[:, :cols].abs() @ K.t())
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, 0, ell, nugget, 0.0, off, rows, 0, cols)
    wb = lib.mplak_kernel_mrhs_workspace_bytes(C.byref(desc), prec, R)
    w = workspace(wb)
    w.fill_(float("nan"))
    _native.check(lib.mplak_kernel_mrhs(C.byref(desc), prec, R, V.data_ptr(), ldv, Y.data_ptr(), ldy, w.data_ptr(), wb,
                                        None, stream()))
    got = host(Y)
    err = np.linalg.norm(got[:, :rows] - ref, axis=1)
    assert np.all(err <= bar * np.linalg.norm(mag, axis=1)) and np.all(got[:, rows:] == 7.0)
