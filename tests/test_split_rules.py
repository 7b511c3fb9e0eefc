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


# A served request's buffer of partials is that of its FP64 products by class; its
# FP32 products in mixed launches are split as far as the same buffer allows.
@pytest.mark.parametrize("n", [1, 64, 300, 1000, 2047, 2048, 4096, 6001, 8000, 8191, 8192, 9999, 12288, 13455, 20000])
@pytest.mark.parametrize("nrhs", [1, 3, 8, 17, 64])
@pytest.mark.parametrize("pairs", [None, "0", "1"])
def test_served_partials_fit_the_fp64_plan(lib, monkeypatch, n, nrhs, pairs):
    from mpla_amd import mpla
    monkeypatch.delenv("MPLAK_RAGGED_PAIRS", raising=False)
    if pairs is not None:
        monkeypatch.setenv("MPLAK_RAGGED_PAIRS", pairs)

    def plan(query, prec):
        s = _native.mplak_ragged_system()
        s.n, s.nrhs, s.dim, s.kind, s.length_scale, s.precision = n, nrhs, 3, 0, 0.5, prec
        return query(C.byref(s)), s

    tiles = -(-n // 512)
    by_class, s = plan(lib.mplak_ragged_plan, F64)
    if pairs == "0" or (pairs is None and n < 8192):
        assert s.scheme == 0 and s.slab_cols % 256 == 0 and by_class == 8 * s.slabs * nrhs * n
    else:
        assert s.scheme == 1 and 0 <= by_class - 8 * 512 * tiles * (tiles + 1) * nrhs <= 8 * tiles * (tiles + 1) + 512
    assert plan(lib.mplak_ragged_plan_mixed, F64)[0] == by_class
    assert 0 < plan(lib.mplak_ragged_plan_mixed, F32)[0] <= by_class
    assert 0 < plan(lambda s: lib.mplak_ragged_plan_within(s, by_class + 300000), F32)[0] <= by_class + 300000
    up = lambda b, to=256: -(-b // to) * to  # noqa: E731
    total = up(24 * n) + 6 * up(8 * n * nrhs) + up(by_class) + up(lib.mplak_ragged_cg_part_bytes(n, nrhs)) + up(8 * n)
    assert mpla.lib().mpla_server_request_bytes(n, 3, nrhs) == up(total, 1 << 20)


# Exact products of few targets and many sources: at least one workgroup (256
# targets, one slab) per CU, and partials that stay within 17 MB.
@pytest.mark.parametrize("rows,cols", [(1, 65536), (256, 65536), (200, 1000000), (257, 65536), (512, 131072),
                                       (1000, 65536), (2048, 65536), (3840, 65535), (3841, 65536), (8192, 65536)])
def test_few_targets_fill_the_chip(lib, rows, cols):
    partials = lib.mplak_kernel_matvec_workspace_bytes(C.byref(desc(rows, cols)))
    slabs = partials // (8 * rows)
    assert -(-rows // 256) * slabs >= 256 and partials <= 17e6


# A plan holds the partial rows of the split its products take: without a
# coincidence shift that of the 16 x 16 tiles (pairs times workgroups below 2400),
# with one that of the vector unit (eight below 820 pairs).
@pytest.mark.parametrize("n", [4096, 8192, 13000, 16000, 19968, 20480, 40000])
def test_plans_hold_the_rows_of_their_split(lib, n):
    tiles = -(-n // 512)
    pairs = tiles * (tiles + 1) // 2
    split = max(k for k in (1, 2, 4, 8) if k == 1 or pairs * k < 2400)
    slots = 4 * -(-tiles // 4)
    plain, shifted = (lib.mplak_screen_plan_bytes(C.byref(desc(n, n, shift=s))) for s in (0.0, 1e-3))
    rows = [max(2 * pairs, tiles * slots * k) for k in (split, 8 if pairs < 820 else 1)]
    assert shifted - plain == (rows[1] - rows[0]) * 512 * 8


# Planning a product of few targets and a million sources: the search for the slab
# count takes microseconds (every count one by one: 150 to 220 us a query).
@pytest.mark.parametrize("rows,prec,R", [(1, F64, 1), (256, F32, 4), (256, BF16, 64), (100, F64, 64)])
def test_planning_is_quick(lib, rows, prec, R):
    import time
    d = desc(rows, 1000000)

    def query():
        t = time.perf_counter()
        lib.mplak_kernel_mrhs_workspace_bytes(C.byref(d), prec, R)
        return time.perf_counter() - t

    assert min(query() for _ in range(100)) < 75e-6
