"""Cholesky above order 64 with an infinite diagonal entry: like in the reference,
its column is zero below it and the columns after it are as if it were not there, so
a later pivot that is negative is still found.  Compared with the oracle; the bound
is that of the finite case, |L L^T| (n + 4) u / (1 - (n + 4) u) per entry of each
factor's product (Higham, Accuracy and Stability, Thm 10.3)."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import _lib, workloads as wl
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
CASES = [(65, 0), (65, 64), (100, 15), (100, 16), (129, 63), (129, 64), (300, 70), (577, 130)]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n,at", CASES)
def test_infinite_pivot(n, at, dt):
    a = wl.spd(n, 7 * n).astype(dt)
    a[at, at] = np.inf
    l = rl.Cholesky.decompose(rl.Matrix(a)).unpack().to_numpy()
    ref = orc.chol_unpack(orc.chol_decompose(a, dtype=dt))
    assert np.array_equal(np.isnan(l), np.isnan(ref)) and np.isnan(l[at, at])
    assert np.all(l[at + 1:, at] == 0)
    keep = np.arange(n) != at
    lk, ak = l[np.ix_(keep, keep)].astype(np.longdouble), a[np.ix_(keep, keep)]
    u = np.finfo(dt).eps / 2
    g = (n + 4) * u / (1 - (n + 4) * u)
    assert np.all(np.abs(ak - lk @ lk.T) <= g * (np.abs(lk) @ np.abs(lk).T))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n,at", [c for c in CASES if c[1] + 1 < c[0]])
def test_failure_after_it(n, at, dt):
    a = wl.spd(n, 9 * n).astype(dt)
    a[at, at] = np.inf
    a[n - 1, n - 1] = -2.0
    with pytest.raises(orc.OracleError):
        orc.chol_decompose(a, dtype=dt)
    with pytest.raises(rl.Error) as e:
        rl.Cholesky.decompose(rl.Matrix(a))
    assert e.value.kind() == rl.ErrorKind.DecompFailure
    assert f"entry {n - 1} " in _lib.last_error()
