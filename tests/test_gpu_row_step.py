"""Swaps, block inverse and block-row solve between the panels of an LU, at the
edges of panels (64), of the columns one workgroup owns (32) and of outer blocks
(512), with swaps that chain.

A = P L U with sparse L (entries 1/2) and U (small integers): every step of the
elimination is exact in FP32 too, and pivot k is the row of L U that P moved, so
the pivots and the factor are known exactly."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import workloads as wl

pytestmark = pytest.mark.gpu


def order(kind, n, r):
    if kind == "up":
        return np.roll(np.arange(n), 1)
    if kind == "down":
        return np.roll(np.arange(n), -1)
    if kind == "reversed":
        return np.arange(n)[::-1].copy()
    return r.permutation(n)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["up", "down", "reversed", "random"])
@pytest.mark.parametrize("n", [65, 66, 95, 96, 97, 127, 128, 129, 161, 511, 512, 513, 545, 577, 641])
def test_exact_factor(n, kind, dt):
    r = wl.rng(n)
    i = np.arange(1, n)
    l = np.eye(n)
    l[i, i // 2] = 0.5
    u = np.diag(2.0 ** r.integers(1, 3, n))
    for d in (1, 3, 40, 70, 200):
        if d < n:
            u += np.diag(r.integers(-2, 3, n - d).astype(float), d)
    p = order(kind, n, r)          # row k of L U is row p[k] of A
    a = np.empty((n, n))
    a[p] = l @ u
    rows, ipiv = np.argsort(p), np.empty(n, dtype=np.int64)
    for k in range(n):
        ipiv[k] = q = k + int(np.flatnonzero(rows[k:] == k)[0])
        rows[[k, q]] = rows[[q, k]]
    f = rl.PartialPivLu.decompose(rl.Matrix(a.astype(dt)))
    assert np.array_equal(f.ipiv(), ipiv)
    assert np.array_equal(f.packed(), (np.tril(l, -1) + u).astype(dt))
