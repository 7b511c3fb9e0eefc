"""Work splits of the kernels at the sizes where they can go wrong: edges of
tiles and panels, remainders, the smallest and largest of a rule's range.
References are plain NumPy or torch in FP64."""
import numpy as np
import pytest

from mpla_amd import _native
from tests.gpu_util import dev, empty, host, require_gpu, stream, workspace

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


@pytest.fixture(scope="module")
def lib():
    require_gpu()
    return _native.mplak()


def ck(status):
    _native.check(status)


# 16-row panels (m n up to 40 MB or m up to 64, n from 256) with their column
# remainders and slabs (n from 4096); 128-row panels otherwise, one slab and
# several; rows that end inside a panel; odd strides and an 8-byte aligned base.
@pytest.mark.parametrize("m,n,lda,shift", [
    (1, 255, 3, 0), (1, 4097, 1, 1), (2, 256, 2, 1), (15, 257, 15, 0), (16, 383, 17, 1), (17, 1030, 17, 0),
    (33, 9001, 35, 1), (64, 4096, 64, 0), (65, 255, 65, 1), (127, 100, 129, 0), (129, 63, 129, 1), (1001, 777, 1001, 1),
    (2200, 2300, 2201, 0), (2301, 2302, 2301, 1), (257, 20011, 257, 0)])
def test_dgemv_panels_slabs_and_strides(lib, m, n, lda, shift):
    rng = np.random.default_rng(m * 7 + n)
    A = rng.uniform(-1, 1, shift + lda * n)
    x = rng.uniform(-1, 1, n + shift)
    A_dev, x_dev, y = dev(A), dev(x), empty(m + 1)
    y.fill_(7.0)
    wb = lib.mplak_dgemv_workspace_bytes(m, n)
    w = workspace(wb)
    ck(lib.mplak_dgemv_f64(m, n, A_dev.data_ptr() + 8 * shift, lda, x_dev.data_ptr() + 8 * shift, y.data_ptr(),
                           w.data_ptr(), wb, None, stream()))
    got = host(y)
    Af = A[shift:].reshape((lda, n), order="F")[:m].astype(np.longdouble)
    xl = x[shift:].astype(np.longdouble)
    # a sum of n products in any order: at most n roundings of a partial sum
    assert np.all(np.abs(got[:m] - Af @ xl) <= (n + 1) * EPS * (np.abs(Af) @ np.abs(xl)))
    assert got[m] == 7.0
