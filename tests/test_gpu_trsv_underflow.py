"""The triangular solves where an entry over its row's diagonal underflows although
its product with the solution does not, and where the solution itself is subnormal.

Bound: |b - M x| <= g |M||x| + |d| s elementwise, g = (n + 8) u / (1 - (n + 8) u)
(substitution's, Higham, Accuracy and Stability, Thm 8.5, with room for the scaled
rows' extra roundings), d the row's diagonal and s the smallest subnormal number: a
quotient below the normal numbers is rounded to a multiple of s."""
import ctypes as C

import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu
N = 140


def holds(m, b, x):
    dt = m.dtype
    u, s = np.finfo(dt).eps / 2, np.finfo(dt).smallest_subnormal
    w = m.astype(np.longdouble)
    x, b = x.astype(np.longdouble), b.astype(np.longdouble)
    g = (len(m) + 8) * u / (1 - (len(m) + 8) * u)
    bound = g * (np.abs(w) @ np.abs(x.T)) + np.abs(np.diag(w))[:, None] * np.longdouble(s)
    return bool(np.all(np.abs(b.T - w @ x.T) <= bound))


def triangular(m, b, upper):
    f = getattr(_lib.load(), f"rlg_solve_{'u' if upper else 'l'}_triangular_{'f64' if m.itemsize == 8 else 'f32'}")
    x, n = np.empty_like(b), len(m)
    assert f(n, n, m.ctypes.data, n, n, len(b), b.ctypes.data, n, x.ctypes.data, n) == 0, _lib.last_error()
    return x


# entry, diagonal and right-hand side: entry / diagonal is 0 or subnormal, the
# solution is normal
LOST = {np.float64: (1.1e-170, 1.3e170, 1e300), np.float32: (1.1e-25, 1.3e25, 1e30)}


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("src,dst", [(0, 1), (0, 63), (65, 127), (128, 139)])
@pytest.mark.parametrize("nrhs", [1, 5, 16])
def test_lost_term(dt, upper, src, dst, nrhs):
    """Row dst takes one term from entry src; the other vectors are ordinary."""
    e, d, v = LOST[dt]
    m = np.eye(N, dtype=dt)
    if upper:
        src, dst = dst, src
    m[dst, src], m[dst, dst] = e, d
    b = wl.rng(dst).standard_normal((nrhs, N)).astype(dt)
    b[nrhs // 2] = 0
    b[nrhs // 2, src] = v
    x = triangular(m, b, upper)
    assert x[nrhs // 2, dst] != 0
    assert holds(m, b, x)


@pytest.mark.parametrize("dt,a,c,v", [(np.float64, 1.3e153, 1e-12, 1e150), (np.float32, 1.3e19, 1e-5, 1e20)])
@pytest.mark.parametrize("at", [0, 62, 64])
@pytest.mark.parametrize("nrhs", [1, 5, 16])
def test_lost_term_transposed(dt, a, c, v, at, nrhs):
    """L^T through a Cholesky factor whose only entry off the diagonal, c / a, lies
    below row `at`, with a^2 on the matrix's diagonal."""
    spd = np.eye(N, dtype=dt)
    spd[at, at], spd[at + 1, at], spd[at, at + 1] = dt(a) * dt(a), c, c
    lib, suf = _lib.load(), "f64" if dt == np.float64 else "f32"
    h, l = C.c_void_p(), np.zeros((N, N), dtype=dt)
    assert getattr(lib, f"rlg_chol_decompose_{suf}")(N, N, spd.ctypes.data, N, C.byref(h)) == 0
    assert getattr(lib, f"rlg_chol_unpack_{suf}")(h, l.ctypes.data, N) == 0
    b = np.zeros((nrhs, N), dtype=dt)
    b[:, at + 1] = v
    x = np.empty_like(b)
    assert getattr(lib, f"rlg_chol_solve_{suf}")(h, N, nrhs, b.ctypes.data, N, x.ctypes.data, N) == 0
    lib.rlg_chol_free(h)
    # the forward solve is exact: b is zero at `at`, and row at + 1's diagonal is 1
    assert l[at + 1, at + 1] == 1 and holds(np.ascontiguousarray(l.T), b, x)


@pytest.mark.parametrize("dt,m,d,y", [(np.float64, -300, 300, -476), (np.float32, -30, 30, -91)])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("size", [0, 1, 40])
def test_subnormal_solution(dt, m, d, y, upper, size):
    """Terms that are each below half the smallest number once divided, together
    above it; and a right-hand side that is (`size`: of that many units)."""
    n = 64
    a = np.eye(n, dtype=dt)
    row = 0 if upper else n - 1
    a[row] = dt(2.0) ** m
    a[row, row] = dt(2.0) ** d
    b = np.full((1, n), dt(2.0) ** y)
    b[0, row] = size * float(np.finfo(dt).smallest_subnormal) * 2.0 ** d * 0.7
    b = b.astype(dt)
    assert holds(a, b, triangular(a, b, upper))


@pytest.mark.parametrize("dt,lo", [(np.float64, -480), (np.float32, -45)])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("n", [64, 128, 193])
def test_wide_range(dt, lo, upper, n):
    """Entries over a wide range of magnitudes, and rows scaled like their diagonals."""
    r = wl.rng(n)
    m = r.choice([-1.0, 1.0], (n, n)) * 2.0 ** r.uniform(lo, 0, (n, n))
    m[np.diag_indices(n)] = 1.0
    m *= 2.0 ** r.uniform(0, -lo, (n, 1))
    m = (np.triu(m) if upper else np.tril(m)).astype(dt)
    b = (np.diag(m) * 2.0 ** r.uniform(lo, 0, (6, n))).astype(dt)
    b[1] = 0
    b[1, n // 2] = np.diag(m)[n // 2]
    assert holds(m, b, triangular(m, b, upper))
