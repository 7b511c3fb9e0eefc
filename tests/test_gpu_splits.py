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


# 16-row panels (m n up to 40 MB and m up to 4096, or m up to 64) with their column
# remainders and slabs (n from 4096); 128-row panels otherwise, one slab and
# several; 32-, 64- and 128-row panels of all columns between (from 128 columns;
# above 8192 rows from 22 MB); rows that end inside a panel; odd strides and an
# 8-byte aligned base.
@pytest.mark.parametrize("m,n,lda,shift", [
    (1, 255, 3, 0), (1, 4097, 1, 1), (2, 256, 2, 1), (15, 257, 15, 0), (16, 383, 17, 1), (17, 1030, 17, 0),
    (33, 9001, 35, 1), (64, 4096, 64, 0), (65, 255, 65, 1), (127, 100, 129, 0), (129, 63, 129, 1), (1001, 777, 1001, 1),
    (2200, 2300, 2201, 0), (2301, 2302, 2301, 1), (257, 20011, 257, 0),
    (226, 208, 226, 0), (4096, 1300, 4097, 1), (4097, 127, 4097, 0), (4097, 128, 4097, 1), (8191, 700, 8193, 0),
    (8193, 300, 8193, 0), (8193, 401, 8193, 1), (16384, 169, 16384, 0), (16385, 337, 16387, 1), (32769, 130, 32769, 0)])
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


# Planned products share a tile pair between 8, 4, 2 and 1 workgroups, by the
# number of 512-point tiles (16, 24, 48 and more); one tile, a ragged last
# tile, unordered points (the vector-unit form) and ordered ones.
@pytest.mark.parametrize("n", [1, 511, 513, 4097, 8192, 8193, 12288, 17000, 25088])
@pytest.mark.parametrize("kind,dim,ordered", [(0, 3, True), (1, 2, True), (0, 2, False), (1, 3, False)])
def test_planned_product_pair_splits(lib, n, kind, dim, ordered):
    import ctypes as C

    import torch
    g = torch.Generator(device="cuda").manual_seed(n + 10 * dim + kind)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    x = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    if ordered:
        perm = torch.empty(n, dtype=torch.int64, device="cuda")
        ob = lib.mplak_spatial_order_workspace_bytes(n, dim)
        ow = workspace(ob)
        ck(lib.mplak_spatial_order(table.data_ptr(), dim, 0, n, perm.data_ptr(), ow.data_ptr(), ob, stream()))
        P = P[:, perm].contiguous()
        table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    ell, nugget = (0.05, 0.1)[kind], 0.75
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, kind, ell, nugget, 0.0, 0, n, 0, n)
    ref, mag = torch.empty_like(x), torch.empty_like(x)
    for i in range(0, n, 4096):
        s = sum((P[d, i:i + 4096, None] - P[d][None, :]) ** 2 for d in range(dim))
        r = (3.0 * s).sqrt() / ell
        k = (-0.5 * s / ell ** 2).exp() if kind == 0 else (1.0 + r) * (-r).exp()
        ref[i:i + 4096], mag[i:i + 4096] = k @ x, k @ x.abs()
    ref += nugget * x
    mag = host(mag + nugget * x.abs())
    y = torch.empty_like(x)
    pb = lib.mplak_screen_plan_bytes(C.byref(desc))
    plan = workspace(pb)
    # dropped entries are below 2^-60 (FP64) and 2^-30 (FP32) and number at most n per row; kept ones carry the
    # entry error of their precision (FP32 2e-5 of the row's sum of magnitudes, FP64 1e-12: the oracle's bars)
    for prec, drop, bar in ((_native.MPLAK_PREC_F64, 60.0, 1e-12), (_native.MPLAK_PREC_F32, 30.0, 2e-5)):
        ck(lib.mplak_screen_plan_build(C.byref(desc), prec, drop, plan.data_ptr(), pb, stream()))
        ck(lib.mplak_kernel_matvec_planned(C.byref(desc), prec, drop, plan.data_ptr(), pb, x.data_ptr(), y.data_ptr(),
                                           None, stream()))
        assert np.all(np.abs(host(y) - host(ref)) <= bar * mag + 0.5 * n * 2.0 ** -drop)


# FP64 multi-right-hand-side products on the matrix cores (from 9 columns):
# rows around the 16-row blocks and 128-row tiles, columns around the 16- and
# 64-column blocks, sources around the 64-point chunks, blocks off the diagonal,
# padded leading dimensions; up to 8 columns, and 5 dimensions, take the vector
# unit, in slabs of 32 sources and more.
@pytest.mark.parametrize("rows,cols,row_off,R,dim", [
    (1, 1, 0, 9, 1), (15, 63, 3, 16, 2), (17, 65, 0, 17, 3), (127, 64, 0, 33, 4), (128, 130, 5, 48, 3),
    (129, 129, 0, 64, 2), (1000, 517, 100, 65, 3), (700, 1500, 0, 73, 2), (300, 300, 0, 8, 3), (300, 300, 0, 20, 5),
    (1, 1, 0, 1, 1), (33, 31, 2, 2, 2), (257, 33, 0, 3, 3), (255, 257, 1, 5, 2), (600, 289, 0, 8, 4), (300, 1000, 5, 24, 5)])
@pytest.mark.parametrize("kind", [0, 1])
def test_mrhs_f64_tiles(lib, rows, cols, row_off, R, dim, kind):
    import ctypes as C

    import torch
    rng = np.random.default_rng(rows + cols + R)
    n = max(cols, row_off + rows)
    P = rng.random((dim, n))
    ell, nugget = (0.3, 0.4)[kind], 0.7
    ldv, ldy = cols + 3, rows + 5
    V = rng.standard_normal((R, ldv))
    s = sum((P[d, row_off:row_off + rows, None] - P[d, None, :cols]) ** 2 for d in range(dim))
    r = np.sqrt(3.0 * s) / ell
    K = np.exp(-0.5 * s / ell ** 2) if kind == 0 else (1.0 + r) * np.exp(-r)
    K[np.arange(row_off, row_off + rows)[:, None] == np.arange(cols)[None, :]] += nugget
    P_dev, V_dev = dev(P), dev(V)
    Y = torch.full((R, ldy), 7.0, dtype=torch.float64, device="cuda")
    table = torch.tensor([P_dev[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, kind, ell, nugget, 0.0, row_off, rows, 0, cols)
    wb = lib.mplak_kernel_mrhs_workspace_bytes(C.byref(desc), _native.MPLAK_PREC_F64, R)
    w = workspace(wb)
    ck(lib.mplak_kernel_mrhs(C.byref(desc), _native.MPLAK_PREC_F64, R, V_dev.data_ptr(), ldv, Y.data_ptr(), ldy,
                             w.data_ptr(), wb, None, stream()))
    got = host(Y)
    # the oracle's FP64 bar: 1e-12 of the sum of magnitudes
    assert np.all(np.abs(got[:, :rows] - V[:, :cols] @ K.T) <= 1e-12 * (np.abs(V[:, :cols]) @ K.T))
    assert np.all(got[:, rows:] == 7.0)


# Multi-right-hand-side products on the matrix cores in lower precision: packed
# blocks of 64 sources (a workgroup stages two at a time), 256-row tiles, one or
# two 32-column blocks, a 64-column group with a narrow rest, several slabs.
@pytest.mark.parametrize("rows,cols,row_off,R,dim", [
    (1, 1, 0, 1, 1), (255, 63, 0, 16, 2), (257, 64, 2, 32, 3), (256, 65, 0, 33, 4), (100, 129, 7, 64, 3),
    (1000, 1537, 100, 65, 3), (1500, 1500, 0, 20, 2), (5000, 4999, 0, 40, 3)])
@pytest.mark.parametrize("prec,bar", [(1, 2e-5), (2, 2e-2), (3, 1e-4)])
def test_mrhs_mfma_blocks(lib, rows, cols, row_off, R, dim, prec, bar):
    import ctypes as C

    import torch
    g = torch.Generator(device="cuda").manual_seed(rows + cols + R)
    n = max(cols, row_off + rows)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    ell, nugget = 0.4, 0.7
    ldv, ldy = cols + 3, rows + 5
    V = torch.randn((R, ldv), generator=g, dtype=torch.float64, device="cuda")
    s = sum((P[d, row_off:row_off + rows, None] - P[d, None, :cols]) ** 2 for d in range(dim))
    r = (3.0 * s).sqrt() / ell
    K = (1.0 + r) * (-r).exp()
    ref, mag = V[:, :cols] @ K.t(), V[:, :cols].abs() @ K.t()
    i = torch.arange(row_off, min(row_off + rows, cols), device="cuda")
    ref[:, i - row_off] += nugget * V[:, i]
    Y = torch.full((R, ldy), 7.0, dtype=torch.float64, device="cuda")
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, 1, ell, nugget, 0.0, row_off, rows, 0, cols)
    wb = lib.mplak_kernel_mrhs_workspace_bytes(C.byref(desc), prec, R)
    w = torch.empty(wb + 8, dtype=torch.uint8, device="cuda")
    for shift in (0, 8):  # a workspace that is 8-byte aligned only
        ck(lib.mplak_kernel_mrhs(C.byref(desc), prec, R, V.data_ptr(), ldv, Y.data_ptr(), ldy, w.data_ptr() + shift, wb,
                                 None, stream()))
        got = host(Y)
        # normwise per column: FP32 entries 2e-5; BF16 operands (8 bits) 2 x 2^-8, split BF16 2^-16 with FP32 sums
        err = np.linalg.norm(got[:, :rows] - host(ref), axis=1)
        assert np.all(err <= bar * np.linalg.norm(host(mag), axis=1) + 1e-30)
        assert np.all(got[:, rows:] == 7.0)


# Exact products around the slab and tile edges of the plain product (square up
# to 2999 points, rectangular blocks, more than 3 dimensions) and of the
# symmetric one, whose tile pairs 8, 4, 2 or 1 workgroups share.
@pytest.mark.parametrize("rows,cols,row_off,dim", [
    (1, 1, 0, 1), (255, 31, 0, 2), (257, 33, 5, 3), (1000, 2049, 7, 3), (2999, 2999, 0, 2), (700, 17000, 0, 3),
    (3000, 3000, 0, 5), (3000, 3000, 0, 1), (3073, 3073, 0, 3), (12289, 12289, 0, 2), (20993, 20993, 0, 3),
    (21505, 21505, 0, 2), (30209, 30209, 0, 3), (42497, 42497, 0, 3)])
@pytest.mark.parametrize("kind,prec,bar", [(0, 0, 1e-12), (1, 0, 1e-12), (1, 1, 2e-5)])
@pytest.mark.parametrize("shift", [0.0, 1e-3])
def test_exact_product_splits(lib, rows, cols, row_off, dim, kind, prec, bar, shift):
    import ctypes as C

    import torch
    if shift and rows > 13000:
        pytest.skip("the coincidence shift takes the same splits; covered at the smaller sizes")
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    n = max(cols, row_off + rows)
    P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
    x = torch.rand(cols, generator=g, dtype=torch.float64, device="cuda") - 0.5
    ell, nugget = 0.3, 0.7
    ref = torch.empty(rows, dtype=torch.float64, device="cuda")
    mag = torch.empty_like(ref)
    for i in range(0, rows, 4096):
        sl = slice(row_off + i, row_off + min(i + 4096, rows))
        s = sum((P[d, sl, None] - P[d][None, :cols]) ** 2 for d in range(dim))
        r = (3.0 * s).sqrt() / ell
        k = (-0.5 * s / ell ** 2).exp() if kind == 0 else (1.0 + r) * (-r).exp()
        k += shift * (s < 1e-28).double()
        k[torch.arange(sl.start, sl.stop, device="cuda")[:, None] == torch.arange(cols, device="cuda")[None]] += nugget
        ref[i:i + 4096], mag[i:i + 4096] = k @ x, k @ x.abs()
    y = torch.full((rows + 1,), 7.0, dtype=torch.float64, device="cuda")
    table = torch.tensor([P[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
    desc = _native.mplak_kernel_desc(table.data_ptr(), dim, kind, ell, nugget, shift, row_off, rows, 0, cols)
    wb = lib.mplak_kernel_matvec_workspace_bytes(C.byref(desc))
    w = torch.empty(wb, dtype=torch.uint8, device="cuda")
    ck(lib.mplak_kernel_matvec(C.byref(desc), prec, x.data_ptr(), y.data_ptr(), w.data_ptr(), wb, None, stream()))
    got = host(y)
    assert np.all(np.abs(got[:rows] - host(ref)) <= bar * host(mag))
    assert got[rows] == 7.0


# Near pairs: chunks around the 64-point groups and 128-row blocks, diagonal pairs
# (symmetric inside), alone and beside far-field items of 1 to 32 terms whose
# columns end inside a wave's pairs of columns.
@pytest.mark.parametrize("am,bm,terms,cols", [(1, 1, 1, 1), (63, 65, 4, 127), (64, 128, 5, 128), (129, 300, 16, 129),
                                              (312, 313, 20, 511), (512, 511, 21, 1025), (500, 512, 32, 300)])
@pytest.mark.parametrize("kind,dim", [(0, 1), (1, 2), (0, 3), (1, 4)])
def test_hmatrix_near_pairs_and_far_items(lib, am, bm, terms, cols, kind, dim):
    import ctypes as C

    import torch
    rng = np.random.default_rng(am * 7 + bm + terms)
    n = max(am + bm, cols + 3)
    P, x = rng.random((dim, n)) * 3.0, rng.standard_normal(n)  # coordinates already scaled
    s = sum((P[d, :, None] - P[d, None, :]) ** 2 for d in range(dim))
    K = np.exp2(-s) if kind == 0 else (1.0 + np.sqrt(s)) * np.exp(-np.sqrt(s))
    V = rng.standard_normal((terms, cols))
    pairs = np.array([[0, am, am, bm], [0, am, 0, am], [am, bm, am, bm]], dtype=np.int64)
    block = np.array([[0, 1, 3, cols, 0, 0]], dtype=np.int64)
    half = cols // 2
    items = np.array([[0, 0, half], [0, half, cols - half]], dtype=np.int64)
    P_dev, x_dev, V_dev = dev(P), dev(x), dev(V)
    pairs_dev, block_dev, items_dev = (torch.as_tensor(v, device="cuda") for v in (pairs, block, items))
    rank = torch.full((1,), terms, dtype=torch.int32, device="cuda")
    part = torch.full((3, 2, 512), 7.0, dtype=torch.float64, device="cuda")
    fpart = torch.full((2, 32), 7.0, dtype=torch.float64, device="cuda")

    class Points(C.Structure):
        _fields_ = [("rows", C.c_void_p), ("cols", C.c_void_p), ("row_ld", C.c_int64), ("col_ld", C.c_int64),
                    ("dim", C.c_int32), ("kind", C.c_int32)]

    pts = Points(P_dev.data_ptr(), P_dev.data_ptr(), n, n, dim, kind)
    for stream_factors in (0, 1):
        ck(lib.mplak_hm_far_near(C.byref(pts), block_dev.data_ptr(), items_dev.data_ptr(), 2, rank.data_ptr(), 32,
                                 V_dev.data_ptr(), x_dev.data_ptr(), fpart.data_ptr(), pairs_dev.data_ptr(), 3,
                                 part.data_ptr(), stream_factors, stream()))
        got, far = host(part), host(fpart)
        a, b = slice(0, am), slice(am, am + bm)
        for k, side, rows, src in ((0, 0, a, b), (0, 1, b, a), (1, 0, a, a), (2, 0, b, b)):
            y, m = K[rows, src] @ x[src], np.abs(K[rows, src]) @ np.abs(x[src])
            assert np.all(np.abs(got[k, side, :y.size] - y) <= 1e-12 * m)  # the oracle's FP64 bar
        for i, cs in enumerate((slice(0, half), slice(half, cols))):
            t, m = V[:, cs] @ x[3:][cs], np.abs(V[:, cs]) @ np.abs(x[3:][cs])
            assert np.all(np.abs(far[i, :terms] - t) <= (cols + 8) * EPS * m)
            assert np.all(far[i, terms:] == 7.0)


# Mixed launches of the served products: pairs from 2048 points on in 8, 4, 2 or 1
# parts, slabs below, every column tile width, every dimension, screened or not;
# each system alone and in the mix gives the same bits.
MIXED = [(1, 2, 0, 1), (63, 3, 1, 3), (700, 1, 0, 2), (2047, 4, 1, 7), (2048, 2, 1, 5), (3000, 3, 0, 8), (5000, 1, 1, 4),
         (9000, 3, 1, 6), (12000, 4, 0, 1), (13000, 2, 0, 3), (18000, 2, 1, 2), (900, 3, 0, 10)]


@pytest.mark.parametrize("drop", [0.0, 30.0])
def test_ragged_mixed_launch(lib, drop):
    import ctypes as C

    import torch
    systems, keep = [], []
    for n, dim, kind, nrhs in MIXED:
        g = torch.Generator(device="cuda").manual_seed(n)
        P = torch.rand((dim, n), generator=g, dtype=torch.float64, device="cuda")
        P = P[:, torch.argsort(P[0])].contiguous()  # some blocks are far apart
        V = torch.randn((nrhs, n), generator=g, dtype=torch.float64, device="cuda")
        Y = torch.full_like(V, 7.0)
        ell = (0.05, 0.1)[kind]
        s = _native.mplak_ragged_system()
        s.points, s.V, s.Y, s.n, s.dim, s.kind, s.nrhs = P.data_ptr(), V.data_ptr(), Y.data_ptr(), n, dim, kind, nrhs
        s.precision, s.length_scale, s.nugget, s.drop_log2 = _native.MPLAK_PREC_F32, ell, 0.75, drop
        part = torch.full((lib.mplak_ragged_plan_mixed(C.byref(s)),), 255, dtype=torch.uint8, device="cuda")  # NaN bits
        s.part = part.data_ptr()
        systems.append(s)
        keep.append((P, V, Y, part, ell))

    def run(members):
        recs = (_native.mplak_ragged_system * len(members))(*[systems[k] for k in members])
        tables = []
        for items_of in (lib.mplak_ragged_product_items, lib.mplak_ragged_finish_items):
            items = []
            for j, k in enumerate(members):
                arr = (_native.mplak_ragged_item * items_of(C.byref(systems[k]), None, j))()
                items_of(C.byref(systems[k]), arr, j)
                items += list(arr)
            tables.append((_native.mplak_ragged_item * len(items))(*items))
        dev_of = lambda a: torch.frombuffer(bytearray(bytes(a)), dtype=torch.uint8).to("cuda")  # noqa: E731
        sd, pd, fd = dev_of(recs), dev_of(tables[0]), dev_of(tables[1])
        ck(lib.mplak_ragged_product_mixed(sd.data_ptr(), pd.data_ptr(), len(tables[0]), stream()))
        ck(lib.mplak_ragged_finish(sd.data_ptr(), fd.data_ptr(), len(tables[1]), stream()))
        return [host(keep[k][2]).copy() for k in members]

    together = run(range(len(MIXED)))
    for k, (n, dim, kind, nrhs) in enumerate(MIXED):
        P, V, _, _, ell = keep[k]
        ref, mag = torch.empty_like(V), torch.empty_like(V)
        for i in range(0, n, 4096):
            s = sum((P[d, i:i + 4096, None] - P[d][None, :]) ** 2 for d in range(dim))
            r = (3.0 * s).sqrt() / ell
            K = (-0.5 * s / ell ** 2).exp() if kind == 0 else (1.0 + r) * (-r).exp()
            ref[:, i:i + 4096], mag[:, i:i + 4096] = V @ K.t(), V.abs() @ K.t()
        bar = 2e-5 * host(mag + 0.75 * V.abs()) + (n * 2.0 ** -drop * host(V.abs().amax()) if drop else 0.0)
        assert np.all(np.abs(together[k] - host(ref + 0.75 * V)) <= bar), MIXED[k]
        assert np.array_equal(run([k])[0], together[k]), MIXED[k]


# One launch per CG iteration up to 6144 elements (2, 4 and 6 per thread of one
# workgroup), three beyond: one iteration of a running column, of one that
# converges in it (its direction is kept), of one that stops at its limit and of
# one that had stopped before (nothing moves).
@pytest.mark.parametrize("n", [1, 63, 1024, 2047, 2048, 2049, 4096, 4097, 6143, 6144, 6145])
@pytest.mark.parametrize("block", [False, True])
def test_cg_iteration_in_one_launch(lib, n, block):
    import ctypes as C
    rng = np.random.default_rng(n)
    cols = 4
    x, r, d, z = (rng.uniform(0.5, 1.5, (cols, n)) for _ in range(4))
    states = (_native.mplak_cg_state * cols)()
    for c, s in enumerate(states):
        s.rr, s.bnorm2, s.n_global, s.eps = float(r[c] @ r[c]), 2.0 * n, n, 1e-30
        s.rule, s.k, s.iter_max, s.done = c & 1, 3, 1000, 0
    states[1].eps, states[2].iter_max, states[3].done = 1e30, 5, 2
    ss = C.sizeof(_native.mplak_cg_state)
    X, R, D, Z = dev(x), dev(r), dev(d), dev(z)
    sin = dev(np.frombuffer(bytes(states), dtype=np.float64).copy())
    sout = dev(np.zeros(cols * ss // 8))
    if block:
        group = dev(np.zeros(8))
        wb = lib.mplak_bcg_workspace_bytes(n, cols)
        w = workspace(wb)
        ck(lib.mplak_bcg_iterate(n, cols, X.data_ptr(), R.data_ptr(), D.data_ptr(), Z.data_ptr(), sin.data_ptr(),
                                 sout.data_ptr(), group.data_ptr(), w.data_ptr(), wb, stream()))
    else:
        wb = lib.mplak_cg_workspace_bytes(n)
        w = workspace(wb)
        for c in range(cols):
            o = 8 * n * c
            ck(lib.mplak_cg_iterate(n, X.data_ptr() + o, R.data_ptr() + o, D.data_ptr() + o, Z.data_ptr() + o,
                                    sin.data_ptr() + ss * c, sout.data_ptr() + ss * c, w.data_ptr(), wb, stream()))
    out = (_native.mplak_cg_state * cols).from_buffer_copy(host(sout).tobytes())
    gx, gr, gd = host(X), host(R), host(D)
    u = (n + 8) * EPS  # any order of n products, then the few operations on the sums
    for c, s in enumerate(states):
        if c == 3:
            assert bytes(out[c]) == bytes(s)
            assert np.array_equal(gx[c], x[c]) and np.array_equal(gr[c], r[c]) and np.array_equal(gd[c], d[c])
            continue
        alpha = s.rr / float(d[c] @ z[c])
        assert abs(out[c].alpha / alpha - 1) <= 2 * u
        rv = r[c] - out[c].alpha * z[c]
        xv = x[c] + out[c].alpha * d[c]
        bound = EPS * 2 * (np.abs(r[c]) + np.abs(out[c].alpha * z[c]))
        assert np.all(np.abs(gr[c] - rv) <= bound)
        assert np.all(np.abs(gx[c] - xv) <= EPS * 2 * (np.abs(x[c]) + np.abs(out[c].alpha * d[c])))
        rr = float(gr[c] @ gr[c])
        assert abs(out[c].rr - rr) <= 2 * u * rr
        rel = np.sqrt(out[c].rr / n) if s.rule == _native.MPLAK_STOP_RMS else np.sqrt(out[c].rr) / np.sqrt(s.bnorm2)
        assert abs(out[c].rel - rel) <= 8 * EPS * rel and out[c].k == 4
        assert out[c].done == (1 if c == 1 else 2 if c == 2 else 0)
        beta = 0.0 if c == 1 else out[c].rr / s.rr
        dv = d[c] if c == 1 else gr[c] + beta * d[c]
        assert np.all(np.abs(gd[c] - dv) <= 4 * EPS * (np.abs(gr[c]) + np.abs(beta * d[c])) * (c != 1))
