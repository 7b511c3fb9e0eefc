"""The workloads whose speed this framework is judged by, each one pass through its public entry points.

Families (a case's "path"):

  dense         y = A x with a stored column-major matrix (mpla_dgemv)
  dense_solve   CG or BiCGSTAB on a stored matrix through the stored-dense core
  product       y = (K + nugget I) x, FP64 kernel entries on the fly (mpla_dgemv_core_kernel_fused)
  block_product Y = K V for a block of right-hand sides in FP64 (mplak_kernel_mrhs)
  solve         mixed-precision kernel solve (mpla_kernel_conjugate_gradient_mixed, FP32 inner products)
  block_solve   multi-right-hand-side kernel solve (mpla_kernel_block_conjugate_gradient_mixed, BF16x3 inner products)
  hmatrix       y = H x with a compressed kernel matrix (mpla_dgemv_core_hmglib_h_matrix); setup belongs to prepare()
  serve         a batch of solve requests in host memory through the server (Server.run_trace)

Points are uniform in the unit cube; kernels are the Gaussian (length scale 0.05) and Matern-3/2 (0.1) of the served
stream, exp(-r^2) for the H-matrix.  Solves run to a relative residual of 1e-10, so that a solution is settled well
below the accuracy of a 1e-9 comparison.
"""
import ctypes as C
import math

import numpy as np
import torch

from mpla_amd import _native, mpla, serving

TOLERANCE = 1e-10
ITER_MAX = 20000
KINDS = {"gaussian": mpla.MPLA_KERNEL_GAUSSIAN, "matern32": mpla.MPLA_KERNEL_MATERN32}
LENGTH = {"gaussian": 0.05, "matern32": 0.1}


def listed():
    return [
        # one dense product small enough that launches and idle CUs decide: the inner step of a small dense solver
        {"name": "dense_1000", "path": "dense", "m": 1000, "n": 1000},
        # a large dense matrix of odd sizes: 4.8 GB streamed from HBM with odd column stride
        {"name": "dense_30001x20003", "path": "dense", "m": 30001, "n": 20003},
        # the dense CG system of the benchmark's size: many short iterations on a cache-resident matrix
        {"name": "dense_cg_4096", "path": "dense_solve", "method": "cg", "n": 4096},
        # a small interpolation operator: the products of an ordinary CG loop at a few thousand points
        {"name": "product_gaussian_3001", "path": "product", "kind": "gaussian", "dim": 3, "n": 3001},
        # an exact product of tens of thousands of unordered points (residual checks, reference solves)
        {"name": "product_matern_40001", "path": "product", "kind": "matern32", "dim": 2, "n": 40001},
        # 64 right-hand sides at once in FP64: the true residuals of a block solve
        {"name": "block_product_20001_r64", "path": "block_product", "kind": "matern32", "dim": 3, "n": 20001, "r": 64},
        # a small interpolation problem solved on its own: latency of a whole solve
        {"name": "solve_matern_4096", "path": "solve", "kind": "matern32", "dim": 2, "n": 4096},
        # the headline system: Gaussian, N = 65536, 3-D, nugget 1
        {"name": "solve_gaussian_65536", "path": "solve", "kind": "gaussian", "dim": 3, "n": 65536},
        # 64 right-hand sides solved together (Matern, nugget 0.5)
        {"name": "block_solve_12000_r64", "path": "block_solve", "kind": "matern32", "dim": 3, "n": 12000, "r": 64},
        # the H-matrix driver's setting: 2-D, exp(-r^2), rank 20, leaves of 512, N = 131072
        {"name": "hmatrix_2d_131072", "path": "hmatrix", "kind": "gaussian", "dim": 2, "n": 131072, "k": 20},
        # a compressed Matern operator in 3-D: near field and far field about equal
        {"name": "hmatrix_3d_40000", "path": "hmatrix", "kind": "matern32", "dim": 3, "n": 40000, "k": 16},
        # a saturated server: twelve ragged requests of 1 to 8 right-hand sides, all there at once
        {"name": "serve_12", "path": "serve", "count": 12, "n_max": 24576, "mix": 1235},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["dense", "dense", "dense_solve", "product", "product", "block_product", "solve", "block_solve",
                       "hmatrix", "hmatrix", "serve"])
    kind = rng.choice(["gaussian", "matern32"])
    dim = rng.choice([2, 3])
    if path == "dense":
        m = _log_int(rng, 64, 30000)
        return {"path": path, "m": m, "n": _log_int(rng, 64, min(30000, 600_000_000 // m))}
    if path == "dense_solve":
        return {"path": path, "method": rng.choice(["cg", "bicgstab"]), "n": _log_int(rng, 300, 8192)}
    if path == "product":
        return {"path": path, "kind": kind, "dim": rng.choice([1, 2, 3, 4]), "n": _log_int(rng, 500, 40000)}
    if path == "block_product":
        return {"path": path, "kind": kind, "dim": dim, "n": _log_int(rng, 1000, 20000), "r": _log_int(rng, 2, 64)}
    if path == "solve":
        return {"path": path, "kind": kind, "dim": dim, "n": _log_int(rng, 1024, 65536)}
    if path == "block_solve":
        return {"path": path, "kind": kind, "dim": dim, "n": _log_int(rng, 1500, 12000), "r": rng.randint(8, 64)}
    if path == "hmatrix":
        return {"path": path, "kind": kind, "dim": dim, "n": _log_int(rng, 10000, 131072 if dim == 2 else 50000),
                "k": rng.randint(8, 24)}
    return {"path": path, "count": rng.randint(2, 12), "n_max": _log_int(rng, 3000, 24576), "mix": rng.randint(1, 9999)}


# ---- inputs: plain torch (numpy for the served requests), from the seed alone


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _uniform(g, *shape, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=g, dtype=torch.float64, device="cuda").mul_(hi - lo).add_(lo)


def _system(case, seed):
    """Points (dim, n) in the unit cube and a block (r, n) of right-hand sides or multiplied vectors."""
    g = _rng(seed)
    points = _uniform(g, case["dim"], case["n"], lo=0.0, hi=1.0)
    return points, torch.randn((case.get("r", 1), case["n"]), generator=g, dtype=torch.float64, device="cuda")


def _length(case):
    # exp(-r^2) for the H-matrix's Gaussian; a Matern of the cube's size, which the far field can compress
    if case["path"] == "hmatrix":
        return 1.0 / math.sqrt(2.0) if case["kind"] == "gaussian" else 1.0
    return LENGTH[case["kind"]]


def _nugget(case):
    if case["path"] in ("hmatrix", "block_product"):
        return 0.0
    return 1.0 if case["kind"] == "gaussian" else 0.5


def _dense_matrix(case, seed):
    """The column-major matrix as a tensor of its columns, and one vector."""
    g = _rng(seed)
    if case["path"] == "dense":
        return _uniform(g, case["n"], case["m"]), _uniform(g, case["n"])
    n = case["n"]
    a = _uniform(g, n, n).mul_(1.0 / math.sqrt(n))
    if case["method"] == "cg":
        a = (a + a.t()) * 0.55  # spectrum in about +-0.9
        a.diagonal().add_(1.0)
    else:
        a.diagonal().add_(_uniform(g, n, lo=2.0, hi=3.0))
    return a.contiguous(), _uniform(g, n)


def _requests(case, seed):
    """The served stream's mix of sizes, kernels and right-hand sides (`mix` says which), with data of the seed."""
    requests = serving.request_stream(case["count"], 1000.0, seed=case["mix"], n_min=1024, n_max=case["n_max"],
                                      tolerance=TOLERANCE)
    rng = np.random.default_rng(int(seed))
    for q in requests:
        q["points"] = rng.random(q["dim"] * q["n"])
        q["rhs"] = rng.standard_normal(q["n"] * q["nrhs"])
    return requests


# ---- the framework's handles, as a program keeps them


class _Session:
    """One instance for the whole program, as the drivers have it."""

    current = None

    def __init__(self):
        self.lib, self.kernels, self.inst = mpla.lib(), _native.mplak(), mpla.mpla_instance()
        self.lib.mpla_init_instance(C.byref(self.inst), mpla.MPI_COMM_WORLD)
        self.inst.verbosity = 0
        self.ref = C.byref(self.inst)
        self.stream = self.lib.mpla_instance_stream(self.ref)

    @classmethod
    def get(cls):
        if cls.current is None:
            cls.current = cls()
        return cls.current


class _Vector:
    """A vector handle on a tensor's memory, as a torch program passes its own vectors."""

    def __init__(self, n, values=None):
        self.s, self.v = _Session.get(), mpla.mpla_vector()
        self.s.lib.mpla_init_vector(C.byref(self.v), self.s.ref, n)
        self.tensor = torch.zeros(n, dtype=torch.float64, device="cuda")
        self.own, self.v.data, self.ref = self.v.data, self.tensor.data_ptr(), C.byref(self.v)
        if values is not None:
            self.tensor.copy_(values)

    def __del__(self):
        self.v.data = self.own
        self.s.lib.mpla_free_vector(self.ref, self.s.ref)


class _Dense:
    def __init__(self, a):
        n, m = a.shape
        self.s, self.a = _Session.get(), mpla.mpla_matrix()
        self.s.lib.mpla_init_matrix(C.byref(self.a), self.s.ref, m, n)
        self.ref = C.byref(self.a)
        _native.check(self.s.kernels.mplak_copy_f64(self.a.data, a.data_ptr(), m * n, self.s.stream))
        self.generic = C.cast(C.pointer(self.a), C.POINTER(mpla.mpla_generic_matrix))
        torch.cuda.synchronize()

    def __del__(self):
        self.s.lib.mpla_free_matrix(self.ref, self.s.ref)


class _Kernel:
    """A matrix-free kernel operator on device points."""

    def __init__(self, case, points):
        self.s, self.points, self.a = _Session.get(), points, mpla.mpla_generic_matrix()
        dim, n = points.shape
        self.table = torch.tensor([points[d].data_ptr() for d in range(dim)], dtype=torch.int64, device="cuda")
        self.data = mpla.mpla_kernel_matrix_data(self.table.data_ptr(), dim, 0, KINDS[case["kind"]], mpla.MPLA_PREC_F64,
                                                 _length(case), _nugget(case), 0.0)
        self.s.lib.mpla_init_generic_matrix(C.byref(self.a), self.s.ref, n, n)
        self.a.data = C.addressof(self.data)
        self.ref = C.byref(self.a)
        d = _native.mplak_kernel_desc()
        d.points, d.dim, d.kind, d.length_scale = self.table.data_ptr(), dim, KINDS[case["kind"]], _length(case)
        d.nugget, d.row_count, d.col_count = _nugget(case), n, n
        self.desc = d

    def __del__(self):
        self.s.lib.mpla_free_generic_matrix(self.ref, self.s.ref)


class _HMatrix:
    def __init__(self, case, points):
        self.s, self.a, self.data = _Session.get(), mpla.mpla_generic_matrix(), mpla.h_matrix_data()
        dim, n = points.shape
        self.s.lib.mpla_init_generic_matrix(C.byref(self.a), self.s.ref, n, n)
        self.ref = C.byref(self.a)
        self.a.data = C.addressof(self.data)
        ptrs = (C.c_void_p * dim)(*[points[d].data_ptr() for d in range(dim)])
        coords = (C.c_void_p * 2)(C.cast(ptrs, C.c_void_p), C.cast(ptrs, C.c_void_p))
        torch.cuda.synchronize()
        self.s.lib.mpla_init_hmatrix_kernel(self.ref, coords, dim, KINDS[case["kind"]], _length(case), _nugget(case),
                                            1.5, 512, case["k"], 0.0, self.s.ref)

    def __del__(self):
        self.s.lib.mpla_destroy_hmglib(self.ref, self.s.ref)
        self.s.lib.mpla_free_generic_matrix(self.ref, self.s.ref)


def prepare(case, seed):
    path, s = case["path"], _Session.get()
    if path == "serve":
        return {"path": path, "requests": _requests(case, seed), "server": serving.Server()}
    if path in ("dense", "dense_solve"):
        a, v = _dense_matrix(case, seed)
        state = {"path": path, "s": s, "a": _Dense(a), "v": _Vector(v.numel(), v), "y": _Vector(a.shape[1])}
        if path == "dense_solve":
            state["core"], state["method"] = mpla.core("mpla_generic_dgemv_core_dense"), case["method"]
        return state
    points, v = _system(case, seed)
    if path == "hmatrix":
        return {"path": path, "s": s, "a": _HMatrix(case, points), "v": _Vector(case["n"], v[0]),
                "y": _Vector(case["n"]), "core": mpla.core("mpla_dgemv_core_hmglib_h_matrix")}
    state = {"path": path, "s": s, "a": _Kernel(case, points), "n": case["n"]}
    if path in ("product", "solve"):
        state.update(v=_Vector(case["n"], v[0]), y=_Vector(case["n"]), core=mpla.core("mpla_dgemv_core_kernel_fused"))
        return state
    state.update(v=v, y=torch.zeros_like(v), r=case["r"])
    if path == "block_product":
        bytes_ = s.kernels.mplak_kernel_mrhs_workspace_bytes(C.byref(state["a"].desc), mpla.MPLA_PREC_F64, case["r"])
        state.update(work=torch.empty(bytes_ // 8 + 1, dtype=torch.float64, device="cuda"), work_bytes=bytes_)
    return state


def run(state):
    path = state["path"]
    if path == "serve":
        return state["server"].run_trace(state["requests"], arrivals=False)[1]
    s, a, v, y = state["s"], state["a"], state["v"], state["y"]
    if path == "dense":
        s.lib.mpla_dgemv(y.ref, a.ref, v.ref, s.ref)
        return y.tensor
    if path == "dense_solve":
        s.lib.mpla_vector_set_zero(y.ref, s.ref)
        solver = (s.lib.mpla_generic_conjugate_gradient_with_checkpoint_restart if state["method"] == "cg"
                  else s.lib.mpla_generic_BiCGSTAB_with_checkpoint_restart)
        solver(v.ref, a.generic, y.ref, ITER_MAX, TOLERANCE, state["core"], 0, False, s.ref)
        return y.tensor
    if path in ("product", "hmatrix"):
        s.lib.mpla_generic_dgemv(y.ref, a.ref, v.ref, state["core"], s.ref)
        return y.tensor
    if path == "solve":
        s.lib.mpla_vector_set_zero(y.ref, s.ref)
        s.lib.mpla_kernel_conjugate_gradient_mixed(v.ref, a.ref, y.ref, ITER_MAX, TOLERANCE, mpla.MPLA_PREC_F32, s.ref)
        return y.tensor
    n, r = state["n"], state["r"]
    if path == "block_product":
        _native.check(s.kernels.mplak_kernel_mrhs(C.byref(a.desc), mpla.MPLA_PREC_F64, r, v.data_ptr(), n, y.data_ptr(),
                                                  n, state["work"].data_ptr(), state["work_bytes"], None, s.stream))
        return y
    y.zero_()
    s.lib.mpla_kernel_block_conjugate_gradient_mixed(v.data_ptr(), y.data_ptr(), r, a.ref, ITER_MAX, TOLERANCE,
                                                     mpla.MPLA_PREC_BF16X3, None, s.ref)
    return y


def work(case):
    """Inputs read once and outputs written once; kernel entries evaluated once per symmetric pair."""
    path = case["path"]
    if path == "serve":
        # n log-uniform up to n_max, 4.5 right-hand sides: about 60 inner products of which the screen keeps a tenth
        mean_n2 = (case["n_max"] ** 2 - 1024 ** 2) / (2.0 * math.log(case["n_max"] / 1024.0))
        return {"bytes": 8.0 * case["count"] * 4.5 * 2.0 * case["n_max"] / 3.0,
                "flops": case["count"] * 60 * 0.1 * mean_n2 * (5.0 + 9.0)}
    n, dim, r = case["n"], case.get("dim", 0), case.get("r", 1)
    entry = 3.0 * dim + 2.0
    if path == "dense":
        return {"bytes": 8.0 * (case["m"] * n + case["m"] + n), "flops": 2.0 * case["m"] * n}
    if path == "dense_solve":
        products = 50 if case["method"] == "cg" else 60  # to 1e-10 on these spectra
        return {"bytes": 8.0 * products * n * n, "flops": 2.0 * products * n * n}
    if path in ("product", "block_product"):
        return {"bytes": 8.0 * n * (dim + 2 * r), "flops": 0.5 * n * n * entry + 2.0 * n * n * r}
    if path == "hmatrix":
        # one level's far blocks hold about 6^(dim - 1) row and column ranges per row; two factors of k terms
        levels = max(1.0, math.log2(n / 512.0))
        terms = 2.0 * case["k"] * n * levels * (3.0 if dim == 2 else 4.0)
        near = min(0.5 * n * n, 0.5 * n * 512.0 * (8 if dim == 2 else 27))
        return {"bytes": 8.0 * terms + 8.0 * n * (dim + 2), "flops": near * (entry + 4.0) + 2.0 * terms}
    products = 60 if path == "solve" else 150
    kept = 0.1 if path == "solve" else 1.0  # the screen of the spatially ordered inner products
    return {"bytes": 8.0 * n * (dim + 2 * r), "flops": products * kept * (0.5 * n * n * entry + 2.0 * n * n * r)}


# ---- 64-bit results in plain torch


def _entries(kind, length, p, q):
    s = torch.zeros((p.shape[1], q.shape[1]), dtype=torch.float64, device="cuda")
    for d in range(p.shape[0]):
        s.add_((p[d][:, None] - q[d][None, :]).square_())
    if kind == "gaussian":
        return s.mul_(-0.5 / length ** 2).exp_()
    s.sqrt_().mul_(math.sqrt(3.0) / length)
    return (1.0 + s) * s.neg().exp_()


def _kernel_times(kind, length, points, v):
    """K v for a block v (r, n), the entries made a slice of rows at a time."""
    n = points.shape[1]
    out = torch.empty_like(v)
    step = max(1, 200_000_000 // n)
    for i in range(0, n, step):
        out[:, i:i + step] = (_entries(kind, length, points[:, i:i + step], points) @ v.t()).t()
    return out


def _solve_spd(a, b):
    """a x = b for a symmetric positive definite a (n, n) and a block b (r, n): CG, restarted once on the residual."""
    def times(v):
        return torch.cat([(a[i:i + 16384] @ v.t()).t() for i in range(0, a.shape[0], 16384)], dim=1)

    x = torch.zeros_like(b)
    for _ in range(2):
        r = b - times(x)
        e, d, rr = torch.zeros_like(b), r.clone(), r.square().sum(1)
        stop = 1e-10 * rr.max().sqrt().item()
        for _ in range(1500):
            z = times(d)
            alpha = torch.where(rr > 0, rr / (d * z).sum(1), 0.0)
            e += alpha[:, None] * d
            r = r - alpha[:, None] * z
            new = r.square().sum(1)
            if new.max().sqrt().item() <= stop:
                break
            d = r + torch.where(rr > 0, new / rr, 0.0)[:, None] * d
            rr = new
        x += e
    return x


def _kernel_solve(kind, length, nugget, points, b):
    n = points.shape[1]
    a = torch.empty((n, n), dtype=torch.float64, device="cuda")
    step = max(1, 200_000_000 // n)
    for i in range(0, n, step):
        a[i:i + step] = _entries(kind, length, points[:, i:i + step], points)
    a.diagonal().add_(nugget)
    return _solve_spd(a, b)


def exact(case, seed):
    path = case["path"]
    if path == "serve":
        out = []
        for q in _requests(case, seed):
            points = torch.as_tensor(q["points"], device="cuda").view(q["dim"], q["n"])
            b = torch.as_tensor(q["rhs"], device="cuda").view(q["nrhs"], q["n"])
            kind = "gaussian" if q["kind"] == mpla.MPLA_KERNEL_GAUSSIAN else "matern32"
            x = _kernel_solve(kind, q["length_scale"], q["nugget"], points, b)
            out.append(np.ascontiguousarray(x.t().cpu().numpy()))
        return out
    if path == "dense":
        a, v = _dense_matrix(case, seed)
        return v @ a
    if path == "dense_solve":
        a, v = _dense_matrix(case, seed)
        return _solve_spd(a, v[None])[0] if case["method"] == "cg" else torch.linalg.solve(a.t().contiguous(), v)
    points, v = _system(case, seed)
    if path in ("solve", "block_solve"):
        x = _kernel_solve(case["kind"], _length(case), _nugget(case), points, v)
        return x if path == "block_solve" else x[0]
    y = _kernel_times(case["kind"], _length(case), points, v) + _nugget(case) * v
    return y if path == "block_product" else y[0]
