"""Pivots of matrices with NaN and infinities: the reference scans from the diagonal
down for a larger magnitude, so a NaN is never taken and one on the diagonal is kept.
The pivots equal the oracle's, in every form of the panel: one workgroup, several, an
order of at most 64, and the batched solver."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import workloads as wl
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def matrices(n):
    r = wl.rng(5 * n)
    a = r.standard_normal((n, n))
    a[[1, n - 2], 3] = [np.inf, -np.inf]
    yield "infinities in two rows", a
    for i, what in ((0, "first"), (n // 2, "middle"), (n - 1, "last")):
        a = r.standard_normal((n, n))
        a[i] = np.nan
        yield f"{what} row", a
        a = r.standard_normal((n, n))
        a[i, i] = np.nan
        yield f"{what} diagonal entry", a
        a = r.standard_normal((n, n))
        a[i, 0] = np.nan
        yield f"{what} entry of the first column", a
    a = r.standard_normal((n, n))
    a[:, 2] = np.nan
    yield "third column", a


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [5, 64, 65, 100, 130, 200, 256, 257, 300, 600, 1100])
def test_pivots(n, dt):
    for what, a in matrices(n):
        a = np.ascontiguousarray(a.astype(dt))
        _, _, ipiv_or = orc.lu_decompose(a, dtype=dt)
        f = rl.PartialPivLu.decompose(rl.Matrix(a))
        assert np.array_equal(f.ipiv(), ipiv_or), what
