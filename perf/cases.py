"""The calls that a program on this library spends its time in, as cases to time.

A case is a dict of plain values; prepare() makes what a program holds before the
call, run() is one pass through the public entry points (the Python classes on
host arrays, or the C ABI on device memory, on the library's own stream), work()
the bytes and operations the call cannot do without, exact() the same results
from numpy or torch in 64 bits.

Operands follow the benchmark's workloads: GEMM U[-1, 1], LU N(0, 1), Cholesky
G G^T / n + I, the refined solve a matrix with singular values log-spaced on
[1, 1e4], the batch half LU and half Cholesky of uneven order.
"""
import ctypes as C
import math

import numpy as np
import torch

import rulinalg_amd as rl
from rulinalg_amd import _lib

DEV = "cuda"
KAPPA = 1e4


def listed():
    return [
        # smallest calls: the order-256 workloads through the host classes, copies included
        {"name": "matmul_host_256", "op": "matmul_host", "m": 256, "k": 256, "n": 256, "dtype": "f64"},
        {"name": "lu_host_256", "op": "factor_host", "kind": "lu", "n": 256, "nrhs": 1, "dtype": "f64"},
        # a small FP32 system with a few right-hand sides, as least squares by normal equations makes them
        {"name": "chol_host_f32_100", "op": "factor_host", "kind": "chol", "n": 100, "nrhs": 3, "dtype": "f32"},
        # an ordinary product of device matrices with ragged sizes (feature matrix times weights)
        {"name": "gemm_f64_1000x777x1283", "op": "gemm", "m": 1000, "k": 777, "n": 1283, "pad": 0, "dtype": "f64"},
        # the FP32 product on the FP32 matrix cores, and the benchmark's large FP64 one
        {"name": "gemm_f32_4096", "op": "gemm", "m": 4096, "k": 4096, "n": 4096, "pad": 0, "dtype": "f32"},
        {"name": "gemm_f64_8192", "op": "gemm", "m": 8192, "k": 8192, "n": 8192, "pad": 0, "dtype": "f64"},
        # one system of the serving mix (log-uniform 16-4096), factored and solved on the device
        {"name": "lu_1531_rhs2", "op": "factor", "kind": "lu", "n": 1531, "nrhs": 2},
        # the same mix's large Cholesky systems
        {"name": "chol_4096_rhs4", "op": "factor", "kind": "chol", "n": 4096, "nrhs": 4},
        # a new right-hand side for a factor kept resident
        {"name": "resolve_lu_4096_rhs1", "op": "resolve", "kind": "lu", "n": 4096, "nrhs": 1},
        # the headline solves at order 16384: plain FP64 with 16 right-hand sides, and refined
        {"name": "lu_16384_rhs16", "op": "factor", "kind": "lu", "n": 16384, "nrhs": 16},
        {"name": "mixed_16384_rhs1", "op": "mixed", "n": 16384, "nrhs": 1},
        # many small systems of uneven order in one launch (a tenth of the benchmark's 20,000)
        {"name": "batch_2000_n8_512", "op": "batch", "count": 2000, "nmax": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matmul_host", "factor_host", "gemm", "gemm", "factor", "factor", "resolve", "mixed", "batch"])
    if op == "matmul_host":
        return {"op": op, "m": _log(rng, 16, 1024), "k": _log(rng, 16, 1024), "n": _log(rng, 16, 1024),
                "dtype": rng.choice(["f64", "f32"])}
    if op == "factor_host":
        kind = rng.choice(["lu", "chol"])
        return {"op": op, "kind": kind, "n": _log(rng, 16, 1024), "nrhs": rng.randint(1, 8),
                "dtype": "f64" if kind == "lu" else rng.choice(["f64", "f32"])}
    if op == "gemm":
        return {"op": op, "m": _log(rng, 64, 8192), "k": _log(rng, 64, 8192), "n": _log(rng, 64, 8192),
                "pad": rng.choice([0, 0, rng.randint(1, 9)]), "dtype": rng.choice(["f64", "f64", "f32", "f32_split"])}
    if op == "factor":
        return {"op": op, "kind": rng.choice(["lu", "chol"]), "n": _log(rng, 128, 10000), "nrhs": rng.randint(1, 16)}
    if op == "resolve":
        return {"op": op, "kind": rng.choice(["lu", "chol"]), "n": _log(rng, 128, 8192), "nrhs": rng.randint(1, 16)}
    if op == "mixed":
        # a product of two factors, as the quick orthogonal matrices of prepare() want it
        return {"op": op, "n": _log(rng, 32, 100) * _log(rng, 32, 100), "nrhs": rng.randint(1, 4)}
    return {"op": op, "count": _log(rng, 50, 2000), "nmax": _log(rng, 16, 512)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, dtype=torch.float64, device=DEV, generator=g)


def _spd(g, n):
    m = _normal(g, n, n)
    a = torch.matmul(m, m.t().contiguous()) / n
    a.diagonal().add_(1.0)
    return a


def _system(case, g):
    """(A, B) of a factor case on the device: B is (nrhs, n), one vector per row."""
    n = case["n"]
    a = _normal(g, n, n) if case["kind"] == "lu" else _spd(g, n)
    return a, _normal(g, case["nrhs"], n)


def _kron_orthogonal(g, n):
    """A dense n x n orthogonal matrix, quickly: the Kronecker product of two random
    orthogonal matrices of orders near sqrt(n), with shuffled rows."""
    p = next(d for d in range(math.isqrt(n), 0, -1) if n % d == 0)
    q = torch.kron(torch.linalg.qr(_normal(g, p, p))[0], torch.linalg.qr(_normal(g, n // p, n // p))[0])
    return q[torch.randperm(n, device=DEV, generator=g)]


def _mixed_system(case, g):
    """A = U diag(s) V^T, s log-spaced on [1, KAPPA] in random order; B = A X."""
    n = case["n"]
    s = torch.logspace(0.0, math.log10(KAPPA), n, dtype=torch.float64, device=DEV)
    s = s[torch.randperm(n, device=DEV, generator=g)]
    a = torch.matmul(_kron_orthogonal(g, n) * s, _kron_orthogonal(g, n).t().contiguous())
    x = _normal(g, case["nrhs"], n)
    return a, torch.matmul(a, x.t().contiguous()).t().contiguous()


def _batch_shapes(case):
    """Orders and right-hand sides of a batch: the case's own, whatever the seed of its values."""
    count = case["count"]
    r = np.random.default_rng([count, case["nmax"]])
    ns = r.integers(8, case["nmax"] + 1, count)
    rs = r.integers(1, 9, count)
    offs = [np.concatenate([[0], np.cumsum(v)]) for v in (ns.astype(np.int64) ** 2, ns.astype(np.int64) * rs, ns.astype(np.int64))]
    return ns, rs, np.arange(count) % 2, offs  # kinds: 0 LU, 1 Cholesky


def _batch_inputs(case, seed):
    ns, rs, kinds, (ao, bo, _) = _batch_shapes(case)
    g = _gen(seed)
    a0 = torch.empty(int(ao[-1]), dtype=torch.float64, device=DEV)
    for n in np.unique(ns):
        for kind in (0, 1):
            idx = np.nonzero((ns == n) & (kinds == kind))[0]
            if len(idx) == 0:
                continue
            m = _normal(g, len(idx), int(n), int(n))
            if kind == 1:
                m = torch.bmm(m, m.transpose(1, 2).contiguous()) / int(n) + torch.eye(int(n), dtype=torch.float64, device=DEV)
            for q, i in enumerate(idx):
                a0[int(ao[i]):int(ao[i + 1])].copy_(m[q].reshape(-1))
    return a0, _normal(g, int(bo[-1]))


class _Lu:
    """A kept factor: the handle and the device matrix it borrows."""

    def __init__(self, kind, a):
        lib = _lib.load()
        self.kind, self.a, self.h = kind, a, C.c_void_p()
        n = a.shape[0]
        f = lib.rlg_lu_decompose_f64_dev if kind == "lu" else lib.rlg_chol_decompose_f64_dev
        _ok(f(n, a.data_ptr(), n, None, C.byref(self.h)))

    def solve(self, b, x):
        lib = _lib.load()
        nrhs, n = b.shape
        f = lib.rlg_lu_solve_f64_dev if self.kind == "lu" else lib.rlg_chol_solve_f64_dev
        _ok(f(self.h, nrhs, b.data_ptr(), n, x.data_ptr(), n, None))

    def pivots(self):
        p = np.empty(self.a.shape[0], dtype=np.int64)
        _ok(_lib.load().rlg_lu_ipiv(self.h, p.ctypes.data))
        return p

    def __del__(self):
        if self.h:
            lib = _lib.load()
            (lib.rlg_lu_free if self.kind == "lu" else lib.rlg_chol_free)(self.h)


def _ok(status):
    if status != 0:
        raise RuntimeError("status %d: %s" % (status, _lib.last_error()))


def prepare(case, seed):
    _lib.load()
    op, g = case["op"], _gen(seed)
    st = {"op": op, "case": case}
    if op in ("matmul_host", "gemm"):
        m, k, n = case["m"], case["k"], case["n"]
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        pad = case.get("pad", 0)  # row strides beyond the columns, as a slice of a wider matrix has
        a = torch.empty(m, k + pad, dtype=dt, device=DEV).uniform_(-1.0, 1.0, generator=g)
        b = torch.empty(k, n + pad, dtype=dt, device=DEV).uniform_(-1.0, 1.0, generator=g)
        if op == "gemm":
            st.update(a=a, b=b, c=torch.zeros(m, n, dtype=dt, device=DEV))
        else:
            st.update(a=rl.Matrix(a.cpu().numpy()), b=rl.Matrix(b.cpu().numpy()))
    elif op == "factor_host":
        a, b = _system(case, g)
        dt = np.float64 if case["dtype"] == "f64" else np.float32
        st.update(a=rl.Matrix(a.cpu().numpy().astype(dt)), b=b.cpu().numpy().astype(dt))
    elif op == "factor":
        a, b = _system(case, g)
        st.update(a0=a, b=b, a=torch.empty_like(a), x=torch.empty_like(b))
    elif op == "resolve":
        a, b = _system(case, g)
        torch.cuda.synchronize()
        st.update(f=_Lu(case["kind"], a), b=b, x=torch.empty_like(b))
    elif op == "mixed":
        a, b = _mixed_system(case, g)
        st.update(a=a, b=b, x=torch.empty_like(b), opts=rl.MixedOptions().to_c())
    else:
        ns, rs, kinds, (ao, bo, po) = _batch_shapes(case)
        a0, b0 = _batch_inputs(case, seed)
        a, b = torch.empty_like(a0), torch.empty_like(b0)
        p = torch.zeros(int(po[-1]), dtype=torch.int64, device=DEV)
        items = (_lib.BatchItem * case["count"])()
        for i in range(case["count"]):
            items[i] = _lib.BatchItem(int(kinds[i]), int(ns[i]), int(rs[i]), -1, a.data_ptr() + 8 * int(ao[i]),
                                      b.data_ptr() + 8 * int(bo[i]), p.data_ptr() + 8 * int(po[i]))
        dev = torch.from_numpy(np.frombuffer(items, dtype=np.uint8).copy()).to(DEV)
        st.update(a0=a0, b0=b0, a=a, b=b, p=p, items=dev,
                  status=dev.view(torch.int32).view(case["count"], -1)[:, 3])
    torch.cuda.synchronize()  # the library works on its own stream
    return st


# ---------------------------------------------------------------- one pass

def run(st):
    lib, case, op = _lib.load(), st["case"], st["op"]
    if op == "matmul_host":
        return (st["a"] * st["b"]).to_numpy()
    if op == "factor_host":
        f = (rl.PartialPivLu if case["kind"] == "lu" else rl.Cholesky).decompose(st["a"])
        return f.solve_many(st["b"])
    if op == "gemm":
        a, b, c = st["a"], st["b"], st["c"]
        f = {"f64": lib.rlg_gemm_f64_dev, "f32": lib.rlg_gemm_f32_dev, "f32_split": lib.rlg_gemm_f32_split_dev}[case["dtype"]]
        _ok(f(case["m"], case["k"], case["n"], 1.0, a.data_ptr(), a.shape[1], b.data_ptr(), b.shape[1], 0.0,
              c.data_ptr(), c.shape[1], None))
        return c
    if op == "factor":
        # the factorization overwrites its matrix: the program keeps the original
        _ok(lib.rlg_dev_copy(st["a"].data_ptr(), st["a0"].data_ptr(), st["a0"].numel() * 8, None))
        f = _Lu(case["kind"], st["a"])
        f.solve(st["b"], st["x"])
        return {"x": st["x"], "packed": st["a"], "ipiv": f.pivots()} if case["kind"] == "lu" else {"x": st["x"]}
    if op == "resolve":
        st["f"].solve(st["b"], st["x"])
        return st["x"]
    if op == "mixed":
        n, rep = st["a"].shape[0], _lib.MixedReport()
        _ok(lib.rlg_solve_mixed_f64_dev(n, st["a"].data_ptr(), n, case["nrhs"], st["b"].data_ptr(), n, st["x"].data_ptr(), n,
                                        C.byref(st["opts"]), C.byref(rep), None))
        return st["x"]
    _ok(lib.rlg_dev_copy(st["a"].data_ptr(), st["a0"].data_ptr(), st["a0"].numel() * 8, None))
    _ok(lib.rlg_dev_copy(st["b"].data_ptr(), st["b0"].data_ptr(), st["b0"].numel() * 8, None))
    _ok(lib.rlg_batch_solve_f64_dev(case["count"], st["items"].data_ptr(), None))
    return {"x": st["b"], "factor": st["a"], "ipiv": st["p"], "status": st["status"]}


# ---------------------------------------------------------------- what a pass cannot do without

def _factor_flops(kind, n, nrhs):
    return (2.0 / 3.0 if kind == "lu" else 1.0 / 3.0) * float(n) ** 3 + 2.0 * float(n) ** 2 * nrhs


def work(case):
    op = case["op"]
    e = 4 if case.get("dtype", "f64").startswith("f32") else 8
    if op in ("matmul_host", "gemm"):
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": e * (m * k + k * n + m * n), "flops": 2.0 * m * k * n}
    if op in ("factor_host", "factor"):
        n, r = case["n"], case["nrhs"]
        return {"bytes": e * (2.0 * n * n + 2.0 * n * r), "flops": _factor_flops(case["kind"], n, r)}
    if op == "resolve":  # each triangle once; Cholesky reads its one triangle for both solves
        n, r = case["n"], case["nrhs"]
        return {"bytes": 8.0 * (n * n * (1.0 if case["kind"] == "lu" else 0.5) + 2.0 * n * r), "flops": 2.0 * n * n * r}
    if op == "mixed":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 8.0 * (n * n + 2.0 * n * r), "flops": _factor_flops("lu", n, r)}
    ns, rs, kinds, (ao, bo, _) = _batch_shapes(case)
    return {"bytes": 8.0 * 2.0 * float(ao[-1] + bo[-1]),
            "flops": float(sum(_factor_flops("lu" if k == 0 else "chol", n, r) for n, r, k in zip(ns, rs, kinds)))}


# ---------------------------------------------------------------- 64-bit results

def exact(case, seed):
    op, g = case["op"], _gen(seed)
    if op in ("matmul_host", "gemm"):
        st = prepare(case, seed)
        m, k, n = case["m"], case["k"], case["n"]
        if op == "matmul_host":
            return np.matmul(st["a"].to_numpy().astype(np.float64), st["b"].to_numpy().astype(np.float64))
        return torch.matmul(st["a"][:, :k].double(), st["b"][:, :n].double())
    if op in ("factor_host", "factor", "resolve"):
        if case["n"] > 6000:
            return None
        a, b = (t.cpu().numpy() for t in _system(case, g))
        if case.get("dtype") == "f32":
            a, b = a.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64)
        x = np.linalg.solve(a, b.T).T.copy()
        return x if op != "factor" else {"x": x, "packed": None, "ipiv": None} if case["kind"] == "lu" else {"x": x}
    if op == "mixed":
        if case["n"] > 6000:
            return None
        a, b = (t.cpu().numpy() for t in _mixed_system(case, g))
        return np.linalg.solve(a, b.T).T.copy()
    ns, rs, kinds, (ao, bo, _) = _batch_shapes(case)
    a0, b0 = (t.cpu().numpy() for t in _batch_inputs(case, seed))
    x = np.empty_like(b0)
    for i, n in enumerate(ns):
        a, b = a0[ao[i]:ao[i + 1]].reshape(n, n), b0[bo[i]:bo[i + 1]].reshape(rs[i], n)
        x[bo[i]:bo[i + 1]] = np.linalg.solve(a, b.T).T.reshape(-1)
    return {"x": x, "factor": None, "ipiv": None, "status": None}
