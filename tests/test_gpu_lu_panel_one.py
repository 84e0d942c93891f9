"""FP64 panels of at most 256 rows, by one workgroup with 1 to 4 rows per lane: at
the edges of those rows, and with a pivot below epsilon in each group of columns."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [66, 127, 128, 130, 191, 192, 193, 254])
def test_row_edges(n):
    """P A = L U to the elementwise bound g |L||U|, g = n u / (1 - n u) (Higham,
    Accuracy and Stability, Thm 9.3) with room for n + 8, and |l| <= 1 up to
    the one rounding of a quotient."""
    a = wl.gaussian(n, n, 5000 + n)
    f = rl.PartialPivLu.decompose(rl.Matrix(a))
    lu, rows = f.packed(), np.arange(n)
    for i, p in enumerate(f.ipiv()):
        rows[[i, p]] = rows[[p, i]]
    l, u = np.tril(lu, -1) + np.eye(n), np.triu(lu)
    assert np.abs(np.tril(lu, -1)).max() <= 1 + 2.0 ** -52
    e = (n + 8) * 2.0 ** -53
    diff = np.abs(l.astype(np.longdouble) @ u.astype(np.longdouble) - a[rows])
    assert np.all(diff <= e / (1 - e) * (np.abs(l) @ np.abs(u)))


@pytest.mark.parametrize("n,j", [(65, 0), (65, 64), (100, 15), (128, 63), (150, 16), (192, 100), (256, 31), (256, 255)])
def test_first_small_pivot(n, j):
    """A zero column stays exactly zero, so its pivot is the first one refused."""
    a = wl.gaussian(n, n, 6000 + n)
    a[:, j] = 0.0
    with pytest.raises(rl.Error, match=r"pivot %d\b" % j):
        rl.PartialPivLu.decompose(rl.Matrix(a))
