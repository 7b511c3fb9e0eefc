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
