"""A NaN pivot: every quotient by it is NaN, whatever is divided, and so is all that
is eliminated with it.  The column holds NaN on the diagonal and zeros elsewhere, so
the pivot is the diagonal's row under any order of candidates."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import workloads as wl
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [64, 65, 130, 200, 257, 600])
@pytest.mark.parametrize("at", [0, 17, 47])
def test_nan_pivot(n, at, dt):
    a = wl.gaussian(n, n, n + at).astype(dt)
    a[:, :at] = np.eye(n, at)
    a[:, at] = 0
    a[at, at] = np.nan
    f = rl.PartialPivLu.decompose(rl.Matrix(a))
    lu_or, _, ipiv_or = orc.lu_decompose(a, dtype=dt)
    assert np.array_equal(f.ipiv(), ipiv_or)
    lu = f.packed()
    assert np.array_equal(np.isnan(lu), np.isnan(lu_or))
    assert np.isnan(lu[at + 1:, at:]).all() and np.array_equal(lu[:at + 1, at + 1:], lu_or[:at + 1, at + 1:])
