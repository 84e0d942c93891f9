"""The triangular solves' sub-block sweep and update at the edges of sub-blocks
(64), steps (128) and right-hand-side groups (4, 8, 16 per launch), and with
values that leave the scaled sweep's range.

Bound: |b - M x| <= (n + 8) u |M||x| / (1 - (n + 8) u) elementwise, substitution's
bound (Higham, Accuracy and Stability, Thm 8.5) with room for the scaled rows'
extra roundings."""
import ctypes as C

import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def solve(m, b, upper):
    lib = _lib.load()
    n, nrhs = m.shape[0], b.shape[0]
    x = np.empty_like(b)
    f = lib.rlg_solve_u_triangular_f64 if upper else lib.rlg_solve_l_triangular_f64
    assert f(n, n, m.ctypes.data, n, n, nrhs, b.ctypes.data, n, x.ctypes.data, n) == 0, _lib.last_error()
    return x


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 193, 257])
def test_sweep(n, upper):
    r = wl.rng(n)
    m = r.standard_normal((n, n)) / np.sqrt(n)
    m[np.diag_indices(n)] = r.uniform(0.5, 2.0, n) * r.choice([-1.0, 1.0], n)
    m = np.triu(m) if upper else np.tril(m)
    for nrhs in (1, 4, 5, 8, 9, 16, 17):
        b = r.standard_normal((nrhs, n))
        x = solve(m, b, upper).astype(np.longdouble)
        g = (n + 8) * U / (1 - (n + 8) * U)
        assert np.all(np.abs(b.T - m.astype(np.longdouble) @ x.T) <= g * (np.abs(m) @ np.abs(x.T)))


@pytest.mark.parametrize("n", [65, 128, 200])
def test_factor_solves(n):
    """L, U and L^T through the factor handles, x apart from b and x = b."""
    lib = _lib.load()
    import torch
    r = wl.rng(7 * n)
    for kind, a in (("lu", r.standard_normal((n, n))), ("chol", wl.spd(n, n))):
        for nrhs in (3, 6, 16):
            b = r.standard_normal((nrhs, n))
            da, db = torch.tensor(a, device="cuda"), torch.tensor(b, device="cuda")
            dx = torch.zeros_like(db)
            torch.cuda.synchronize()
            h = C.c_void_p()
            assert getattr(lib, f"rlg_{kind}_decompose_f64_dev")(n, da.data_ptr(), n, None, C.byref(h)) == 0
            f = getattr(lib, f"rlg_{kind}_solve_f64_dev")
            assert f(h, nrhs, db.data_ptr(), n, dx.data_ptr(), n, None) == 0
            assert f(h, nrhs, db.data_ptr(), n, db.data_ptr(), n, None) == 0
            assert lib.rlg_synchronize() == 0
            getattr(lib, f"rlg_{kind}_free")(h)
            assert torch.equal(dx, db)
            x = dx.cpu().numpy()
            eta = np.abs(b.T - a @ x.T).max() / (np.abs(a).sum(1).max() * np.abs(x).max())
            assert eta <= 1e-13


@pytest.mark.parametrize("at", [1, 63, 64, 127, 130])
def test_outside_the_scaled_range(at):
    """A row whose entries over its diagonal overflow although the solution does
    not, and an infinite right-hand side: entries before it stay finite."""
    n = 140
    m = np.eye(n)
    m[at, 0], m[at, at] = 1e300, 1e-12
    b = np.zeros((1, n))
    b[0, 0], b[0, at] = 1e-305, 1e-5 + 1e-13
    x = solve(m, b, False)
    assert x[0, 0] == 1e-305 and np.isfinite(x).all()
    assert abs(x[0, at] - 0.1) <= 1e-3  # 1e-13 / 1e-12, with 1e-5's rounding
    b = np.ones((1, n))
    b[0, at] = np.inf
    x = solve(np.tril(np.ones((n, n))), b, False)
    assert np.isfinite(x[0, :at]).all() and x[0, at] == np.inf
    x = solve(np.triu(np.ones((n, n))), b, True)
    assert np.isfinite(x[0, at + 1:]).all() and x[0, at] == np.inf
