"""Block columns of orders above 64 (16-column panels) at the edges of panels
and blocks.  Bound: |A - L L^T| <= g |L||L^T| elementwise, g = (n + 4) u / (1 -
(n + 4) u) (Higham, Accuracy and Stability, Thm 10.3, with room for the
square roots and quotients being good to an ulp instead of half of one)."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [65, 79, 80, 81, 95, 112, 127, 128, 129, 191, 193, 577])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 60])
def test_block_columns(n, dt, scale):
    a = (wl.spd(n, 40 + n) * scale).astype(dt)
    l = rl.Cholesky.decompose(rl.Matrix(a)).unpack().to_numpy()
    assert l.dtype == dt and np.all(np.triu(l, 1) == 0)
    lw = l.astype(np.longdouble)
    u = np.finfo(dt).eps / 2
    g = (n + 4) * u / (1 - (n + 4) * u)
    assert np.all(np.abs(a - lw @ lw.T) <= g * (np.abs(lw) @ np.abs(lw).T))


@pytest.mark.parametrize("n,at", [(65, 0), (70, 15), (100, 16), (129, 63), (129, 64), (200, 199)])
def test_first_failing_column(n, at):
    a = wl.spd(n, 90 + n)
    a[at, at] = -2.0
    a[n - 1, n - 1] = -2.0
    with pytest.raises(rl.Error) as e:
        rl.Cholesky.decompose(rl.Matrix(a))
    assert e.value.kind() == rl.ErrorKind.DecompFailure
    assert f"entry {at} " in _lib.last_error()
