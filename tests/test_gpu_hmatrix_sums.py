"""Rows of an H-matrix product from given factors and near partials, through the
kernel ABI, against NumPy."""
import ctypes as C

import numpy as np
import pytest

from mpla_amd import _native
from tests.gpu_util import dev, host, require_gpu

pytestmark = pytest.mark.gpu


class Chunk(C.Structure):
    _fields_ = [("leaf", C.c_int32), ("count", C.c_int32), ("r0", C.c_int64)]


@pytest.fixture(scope="module")
def lib():
    require_gpu()
    return _native.mplak()


class Rows:
    """`leaves` row leaves of `m` rows with `far` admissible blocks of `rank` terms and
    `ents` near partials each."""

    def __init__(self, leaves, m, far, rank, ents):
        import torch
        rng = np.random.default_rng(m * 5 + far)
        n, nb = leaves * m, leaves * far
        self.n, self.nchunks, self.kmax = n, leaves * -(-m // 128), rank
        U, t = rng.standard_normal((nb, rank, m)), rng.standard_normal((nb, rank))
        part, ent = rng.standard_normal((leaves * ents, 512)), rng.permutation(leaves * ents)
        blocks = np.array([(b // max(far, 1) * m, m, 0, m, b * rank * m, 0) for b in range(nb)], dtype=np.int64)
        chunks = [(leaf, min(128, m - r), leaf * m + r) for leaf in range(leaves) for r in range(0, m, 128)]
        near = part[ent][:, :m].reshape(leaves, ents, m).astype(np.longdouble).sum(1)
        farv = (U.astype(np.longdouble) * t[:, :, None]).reshape(leaves, far * rank, m).sum(1)
        self.ref = (near + farv).reshape(-1)
        self.mag = (np.abs(part[ent][:, :m]).reshape(leaves, ents, m).sum(1)
                    + (np.abs(U) * np.abs(t)[:, :, None]).reshape(leaves, far * rank, m).sum(1)).reshape(-1)
        ints = lambda a, d=np.int64: torch.as_tensor(np.ascontiguousarray(a, dtype=d), device="cuda")  # noqa: E731
        self.chunks = torch.frombuffer(bytearray(bytes((Chunk * len(chunks))(*chunks))), dtype=torch.uint8).to("cuda")
        self.chunk_near, self.near_start = ints([c[0] for c in chunks]), ints(np.arange(leaves) * m)
        self.ent_ptr, self.ent, self.part = ints(np.arange(leaves + 1) * ents), ints(ent), dev(part)
        self.far_ptr, self.far_blk = ints(np.arange(leaves + 1) * far), ints(np.arange(nb), np.int32)
        self.blocks, self.rank = ints(blocks), ints(np.full(nb, rank), np.int32)
        self.U, self.t, self.ys = dev(U), dev(t), dev(np.full(n + 1, 7.0))


def p(t):
    return t.data_ptr()


@pytest.mark.parametrize("leaves,m,far,rank,ents", [(3, 512, 4, 20, 9), (2, 65, 0, 8, 1), (5, 129, 11, 32, 0),
                                                    (40, 1, 9, 1, 3), (2, 313, 17, 7, 20)])
def test_apply_pairs_in_one_launch(lib, leaves, m, far, rank, ents):
    import torch
    r = Rows(leaves, m, far, rank, ents)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    graph, count = C.c_void_p(), C.c_size_t()
    assert lib.hipStreamBeginCapture(C.c_void_p(s.cuda_stream), 2) == 0  # relaxed
    status = lib.mplak_hm_apply_pairs(p(r.chunks), r.nchunks, p(r.chunk_near), p(r.near_start), p(r.ent_ptr), p(r.ent),
                                      p(r.part), p(r.far_ptr), p(r.far_blk), p(r.blocks), p(r.rank), r.kmax, p(r.U),
                                      p(r.t), p(r.ys), s.cuda_stream)
    assert lib.hipStreamEndCapture(C.c_void_p(s.cuda_stream), C.byref(graph)) == 0 and status == 0
    assert lib.hipGraphGetNodes(graph, None, C.byref(count)) == 0 and count.value == 1
    assert lib.hipGraphDestroy(graph) == 0
    _native.check(lib.mplak_hm_apply_pairs(p(r.chunks), r.nchunks, p(r.chunk_near), p(r.near_start), p(r.ent_ptr),
                                           p(r.ent), p(r.part), p(r.far_ptr), p(r.far_blk), p(r.blocks), p(r.rank),
                                           r.kmax, p(r.U), p(r.t), p(r.ys), torch.cuda.current_stream().cuda_stream))
    got = host(r.ys)
    # a sum in any order: at most one rounding of a partial sum per term
    assert np.all(np.abs(got[:-1] - r.ref) <= (far * rank + ents) * 2.0 ** -53 * r.mag) and got[-1] == 7.0


def median_us(f, runs=15):
    import torch
    times = []
    for _ in range(runs):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 1e3)
    return sorted(times)[runs // 2]


# The per-row product with stored near entries reads 2 GB of them once: it keeps at
# least three quarters of the rate of a plain sum of the same buffer, so its far
# field may not take the registers that its resident waves need.
def test_stored_near_entries_stream(lib):
    import torch
    m, leaves, ranges = 512, 256, 4
    n = m * leaves
    g = torch.Generator(device="cuda").manual_seed(3)
    st = torch.rand((leaves, ranges, m, m), generator=g, dtype=torch.float64, device="cuda") - 0.5  # column-major blocks
    xs = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") - 0.5
    ys = torch.full((n + 1,), 7.0, dtype=torch.float64, device="cuda")
    col = [[(leaf + 3 * k) % leaves for k in range(ranges)] for leaf in range(leaves)]
    ints = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.int64), device="cuda")  # noqa: E731
    chunks = (Chunk * (n // 128))(*[(r // m, 128, r) for r in range(0, n, 128)])
    chunks = torch.frombuffer(bytearray(bytes(chunks)), dtype=torch.uint8).to("cuda")
    leaf_range, near_ptr = ints([(leaf * m, m) for leaf in range(leaves)]), ints(np.arange(leaves + 1) * ranges)
    near_cols = ints([(c * m, m) for row in col for c in row])
    near_off, far_ptr = ints(np.arange(leaves * ranges) * m * m), ints(np.zeros(leaves + 1))

    def product():
        _native.check(lib.mplak_hm_apply_stored(p(chunks), n // 128, p(leaf_range), p(near_ptr), p(near_cols),
                                                p(near_off), p(st), p(far_ptr), None, None, None, 1, None, None, p(xs),
                                                p(ys), torch.cuda.current_stream().cuda_stream))

    product()
    ref = torch.stack([(st[leaf] * xs.view(leaves, m)[col[leaf]][:, :, None]).sum((0, 1)) for leaf in range(leaves)])
    assert float((ys[:-1] - ref.reshape(-1)).abs().max()) <= 1e-12 * ranges * m and float(ys[-1]) == 7.0
    assert median_us(product) <= median_us(lambda: st.sum()) / 0.75
