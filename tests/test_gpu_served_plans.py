"""Products of served systems as mplak_ragged_plan_mixed plans them: FP32 in a
mixed launch, FP64 by class, against torch in FP64."""
import ctypes as C

import numpy as np
import pytest

from mpla_amd import _native
from tests.gpu_util import host, require_gpu, stream

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    require_gpu()
    return _native.mplak()


# Slabs of one chunk (FP32 partials of FP32 products) and longer ones, pairs in
# 4, 2 and 1 parts, pairs that the buffer does not hold (6000 points, 64 columns),
# column tiles with a rest.
@pytest.mark.parametrize("n,dim,nrhs", [(1, 1, 1), (65, 2, 3), (700, 3, 5), (2047, 4, 9), (2048, 1, 2), (2300, 2, 64),
                                        (5000, 3, 10), (6000, 2, 64), (8191, 4, 1), (8192, 3, 4), (12000, 1, 1),
                                        (17500, 2, 2)])
@pytest.mark.parametrize("prec,bar", [(_native.MPLAK_PREC_F32, 2e-5), (_native.MPLAK_PREC_F64, 1e-12)])
@pytest.mark.parametrize("kind,drop", [(0, 0.0), (1, 45.0)])
def test_served_products(lib, n, dim, nrhs, prec, bar, kind, drop):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    P = P[:, torch.argsort(P[0])].contiguous()  # some blocks are far apart
    V = torch.randn((nrhs, n), generator=g, dtype=torch.float64, device="cuda")
    Y = torch.full_like(V, 7.0)
    ell = (0.05, 0.1)[kind]
    s = _native.mplak_ragged_system()
    s.points, s.V, s.Y, s.n, s.dim, s.kind, s.nrhs = P.data_ptr(), V.data_ptr(), Y.data_ptr(), n, dim, kind, nrhs
    s.precision, s.length_scale, s.nugget, s.drop_log2 = prec, ell, 0.75, drop
    part = torch.full((lib.mplak_ragged_plan_mixed(C.byref(s)) + 64,), 255, dtype=torch.uint8, device="cuda")  # NaN bits
    s.part = part.data_ptr()
    tables = []
    for items_of in (lib.mplak_ragged_product_items, lib.mplak_ragged_finish_items):
        arr = (_native.mplak_ragged_item * items_of(C.byref(s), None, 0))()
        items_of(C.byref(s), arr, 0)
        tables.append(arr)
    sd, pd, fd = (torch.frombuffer(bytearray(bytes(a)), dtype=torch.uint8).to("cuda") for a in (s, *tables))
    if prec == _native.MPLAK_PREC_F32:
        _native.check(lib.mplak_ragged_product_mixed(sd.data_ptr(), pd.data_ptr(), len(tables[0]), stream()))
    else:
        _native.check(lib.mplak_ragged_product(sd.data_ptr(), pd.data_ptr(), len(tables[0]), s.rt, dim, prec, s.scheme,
                                               stream()))
    _native.check(lib.mplak_ragged_finish(sd.data_ptr(), fd.data_ptr(), len(tables[1]), stream()))
    got = host(Y)
    ref, mag = torch.empty_like(V), torch.empty_like(V)
    for i in range(0, n, 4096):
        d2 = sum((P[d, i:i + 4096, None] - P[d][None, :]) ** 2 for d in range(dim))
        r = (3.0 * d2).sqrt() / ell
        K = (-0.5 * d2 / ell ** 2).exp() if kind == 0 else (1.0 + r) * (-r).exp()
        ref[:, i:i + 4096], mag[:, i:i + 4096] = V @ K.t(), V.abs() @ K.t()
    dropped = n * 2.0 ** -drop * host(V.abs().amax()) if drop else 0.0
    assert np.all(np.abs(got - host(ref + 0.75 * V)) <= bar * host(mag + 0.75 * V.abs()) + dropped)
    assert np.all(host(part)[-64:] == 255)
