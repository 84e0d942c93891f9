"""Host operands whose rows are not contiguous: the gaps are neither read nor
written, also where the rows are moved in more than one piece (32 MB each)."""
import ctypes as C

import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu
NAN = float("nan")


def strided(a, pad):
    """A copy of `a` in rows `pad` longer, the gaps NaN."""
    s = np.full((a.shape[0], a.shape[1] + pad), NAN)
    s[:, :a.shape[1]] = a
    return s


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (1, 5, 7), (3, 2, 1), (67, 33, 130)])
def test_gemm(m, k, n):
    lib = _lib.load()
    r = wl.rng(m + n)
    a = r.integers(-8, 9, (m, k)).astype(float)
    b = r.integers(-8, 9, (k, n)).astype(float)
    for pa, pb, pc in ((0, 0, 3), (2, 0, 0), (0, 5, 1), (1, 2, 3)):
        sa, sb, sc = strided(a, pa), strided(b, pb), np.full((m, n + pc), NAN)
        assert lib.rlg_gemm_f64(m, k, sa.ctypes.data, k + pa, k, n, sb.ctypes.data, n + pb,
                                sc.ctypes.data, n + pc) == 0, _lib.last_error()
        assert np.array_equal(sc[:, :n], a @ b)
        assert np.isnan(sc[:, n:]).all()


def test_pieces():
    """2100 rows of 16.8 KB: two pieces up and down."""
    n, pad, lib = 2100, 3, _lib.load()
    a = wl.spd(n, 5)
    sa, sl = strided(a, pad), np.full((n, n + pad), NAN)
    tight, h = np.zeros((n, n)), C.c_void_p()
    assert lib.rlg_chol_decompose_f64(n, n, sa.ctypes.data, n + pad, C.byref(h)) == 0, _lib.last_error()
    assert lib.rlg_chol_unpack_f64(h, sl.ctypes.data, n + pad) == 0
    assert lib.rlg_chol_unpack_f64(h, tight.ctypes.data, n) == 0
    assert lib.rlg_chol_unpack_f64(h, tight.ctypes.data, n - 1) != 0  # rows would overlap
    lib.rlg_chol_free(h)
    assert np.array_equal(sl[:, :n], tight) and np.isnan(sl[:, n:]).all()
    # substitution-free check: |L L^T - A| <= (n + 2) u |L||L^T| (Higham, Thm 10.3)
    l = np.tril(tight)
    assert np.all(np.abs(l @ l.T - a) <= 2 * (n + 2) * 2.0 ** -53 * (np.abs(l) @ np.abs(l.T)))


@pytest.mark.parametrize("n", [1, 2, 65, 300])
def test_diagonal(n):
    """Diagonal (LU of an upper triangular matrix of powers of two: exact) and
    strided right-hand sides."""
    r = wl.rng(n)
    d = 2.0 ** r.integers(-1, 2, n)
    a = np.tril(r.integers(-1, 2, (n, n)).astype(float), -1) * 0.25
    a[np.diag_indices(n)] = d
    u = np.triu(a.T)  # upper triangular: no row is exchanged, U = u
    m = rl.Matrix(u)
    want = float(np.prod(d))
    assert rl.PartialPivLu.decompose(m).det() == want
    f, p = rl.FullPivLu.decompose(m), 1.0
    for v in np.diag(f.unpack().u.to_numpy()):
        p *= v
    assert abs(f.det()) == abs(p)
    lib, h = _lib.load(), C.c_void_p()
    assert lib.rlg_lu_decompose_f64(n, n, u.ctypes.data, n, C.byref(h)) == 0
    b = r.standard_normal((3, n))
    sb, sx, x = strided(b, 2), np.full((3, n + 4), NAN), np.zeros((3, n))
    assert lib.rlg_lu_solve_f64(h, n, 3, sb.ctypes.data, n + 2, sx.ctypes.data, n + 4) == 0
    assert lib.rlg_lu_solve_f64(h, n, 3, b.ctypes.data, n, x.ctypes.data, n) == 0
    lib.rlg_lu_free(h)
    assert np.array_equal(sx[:, :n], x) and np.isnan(sx[:, n:]).all()
