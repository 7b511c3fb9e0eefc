"""Work splits that need no GPU: the workspace queries tell how many slabs of
sources a product is cut into."""
import ctypes as C

import pytest

from mpla_amd import _native

F64, F32, BF16, BF16X3 = (_native.MPLAK_PREC_F64, _native.MPLAK_PREC_F32, _native.MPLAK_PREC_BF16,
                          _native.MPLAK_PREC_BF16X3)


@pytest.fixture(scope="module")
def lib():
    return _native.mplak()


def desc(rows, cols, dim=3, kind=1, shift=0.0):
    # the points are not read by the queries
    return _native.mplak_kernel_desc(0x1000, dim, kind, 0.3, 0.5, shift, 0, rows, 0, cols)


# The matrix cores add a slab up in FP32: no slab is longer than the share of one
# of 2048 workgroups of 256 targets, in whole 256-source chunks.
@pytest.mark.parametrize("prec", [F32, BF16, BF16X3])
@pytest.mark.parametrize("rows,cols", [(1, 100000), (300, 256), (3000, 3000), (6000, 6000), (9000, 9000), (11521, 11521),
                                       (12000, 12000), (16000, 16000), (20001, 20001), (30000, 30000), (50000, 50000),
                                       (131072, 131072), (2500, 20000), (20000, 2500), (262144, 999)])
@pytest.mark.parametrize("R", [16, 40, 64])
def test_fp32_sums_of_block_products_stay_short(lib, prec, rows, cols, R):
    tiles, chunks = -(-rows // 256), -(-cols // 256)
    longest = 256 * -(-chunks // min(chunks, -(-2048 // tiles)))
    # packed sources (coordinates, then 8 operands of 64 lanes per 16 sources and
    # 32 columns), then a column of FP32 partials per slab and right-hand side
    ops = 4 * -(-R // 32) * 64 * (32 if prec == F32 else 16) * (2 if prec == BF16X3 else 1)
    packed = -(-(-(-cols // 64) * (64 * 16 + ops) + 16) // 256) * 256
    slabs = (lib.mplak_kernel_mrhs_workspace_bytes(C.byref(desc(rows, cols)), prec, R) - packed) // (4 * R * rows)
    assert slabs * longest >= cols
