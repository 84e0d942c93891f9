"""The LU panel at the edges of its 16-column groups, workgroups (256 rows in
FP64, 512 in FP32) and panels, and with an exact tie at every step."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import workloads as wl
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 79, 80, 81, 129, 255, 256, 257, 273, 511, 513])
def test_panel_edges(n):
    """P A = L U to the elementwise bound g |L||U|, g = n u / (1 - n u) (Higham,
    Accuracy and Stability, Thm 9.3) with room for n + 8, and |l| <= 1 up to
    the one rounding of a quotient."""
    a = wl.gaussian(n, n, 3000 + n)
    f = rl.PartialPivLu.decompose(rl.Matrix(a))
    lu, rows = f.packed(), np.arange(n)
    for i, p in enumerate(f.ipiv()):
        rows[[i, p]] = rows[[p, i]]
    l, u = np.tril(lu, -1) + np.eye(n), np.triu(lu)
    assert np.abs(np.tril(lu, -1)).max() <= 1 + 2.0 ** -52
    e = (n + 8) * 2.0 ** -53
    diff = np.abs(l.astype(np.longdouble) @ u.astype(np.longdouble) - a[rows])
    assert np.all(diff <= e / (1 - e) * (np.abs(l) @ np.abs(u)))


def hadamard(n):
    h = np.ones((1, 1))
    while h.shape[0] < n:
        h = np.block([[h, h], [h, -h]])
    return h


@pytest.mark.parametrize("n,dt", [(64, np.float64), (256, np.float64), (512, np.float64), (1024, np.float64),
                                  (512, np.float32), (1024, np.float32)])
def test_exact_ties(n, dt):
    """A Sylvester matrix with shuffled rows: every step's candidates are powers
    of two and tie, and elimination is exact, so the pivots and the factor equal
    the oracle's."""
    a = hadamard(n)[wl.rng(n).permutation(n)].astype(dt)
    f = rl.PartialPivLu.decompose(rl.Matrix(a))
    lu_or, _, ipiv_or = orc.lu_decompose(a, dtype=dt) if dt == np.float32 else orc.lu_decompose(a)
    assert np.array_equal(f.ipiv(), ipiv_or)
    assert np.array_equal(f.packed(), lu_or)
