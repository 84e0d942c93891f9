"""The triangular solves' loads of whole blocks (128 columns) and row groups (64),
next to partial ones, for aligned and unaligned rows.

Bounds, elementwise with g(k) = k u / (1 - k u): g(n + 8) |M||x| for one solve
(Higham, Accuracy and Stability, Thm 8.5), g(3 n + 16) |L||L^T||x| for a Cholesky
solve (Thm 10.4, the factor's error included)."""
import ctypes as C

import numpy as np
import pytest

from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu


def g(k):
    return k * 2.0 ** -53 / (1 - k * 2.0 ** -53)


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("n", [191, 192, 194, 256, 320, 383, 386])
def test_one_solve(n, upper):
    lib, r = _lib.load(), wl.rng(40 + n)
    m = r.standard_normal((n, n)) / np.sqrt(n)
    m[np.diag_indices(n)] = r.uniform(0.5, 2.0, n) * r.choice([-1.0, 1.0], n)
    m = np.triu(m) if upper else np.tril(m)
    f = lib.rlg_solve_u_triangular_f64 if upper else lib.rlg_solve_l_triangular_f64
    for nrhs in (1, 4, 5, 16):
        b = r.standard_normal((nrhs, n))
        x = np.empty_like(b)
        assert f(n, n, m.ctypes.data, n, n, nrhs, b.ctypes.data, n, x.ctypes.data, n) == 0, _lib.last_error()
        x = x.astype(np.longdouble)
        assert np.all(np.abs(b.T - m.astype(np.longdouble) @ x.T) <= g(n + 8) * (np.abs(m) @ np.abs(x.T)))


@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("n", [192, 257, 320, 386])
def test_cholesky_solve(n, pad):
    import torch
    lib, a = _lib.load(), wl.spd(n, 50 + n)
    l = np.abs(np.linalg.cholesky(a))
    for nrhs in (1, 4, 5, 16):
        b = wl.rng(60 + n).standard_normal((nrhs, n))
        da = torch.zeros((n, n + pad), device="cuda", dtype=torch.float64)
        da[:, :n] = torch.tensor(a)
        db = torch.tensor(b, device="cuda")
        dx = torch.zeros_like(db)
        torch.cuda.synchronize()
        h = C.c_void_p()
        assert lib.rlg_chol_decompose_f64_dev(n, da.data_ptr(), n + pad, None, C.byref(h)) == 0
        assert lib.rlg_chol_solve_f64_dev(h, nrhs, db.data_ptr(), n, dx.data_ptr(), n, None) == 0
        assert lib.rlg_synchronize() == 0
        torch.cuda.synchronize()
        lib.rlg_chol_free(h)
        x = dx.cpu().numpy().astype(np.longdouble)
        assert np.all(np.abs(b.T - a.astype(np.longdouble) @ x.T) <= g(3 * n + 16) * (l @ (l.T @ np.abs(x.T))))
