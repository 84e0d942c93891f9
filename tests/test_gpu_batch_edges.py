"""Batched systems at the edges of panels (8, 16), tiles (16), strips (128) and
rows per thread (256), with swaps that chain.

L, U and the Cholesky factor are sparse with halves and powers of two, and the
solutions small integers, so every step is exact: pivots, factors and solutions
are known."""
import numpy as np
import pytest

from rulinalg_amd import batch, workloads as wl

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129, 143, 144, 145, 255, 256, 257, 272, 273, 385,
         511, 512]


def order(kind, n, r):
    if kind == "up":
        return np.roll(np.arange(n), 1)
    if kind == "down":
        return np.roll(np.arange(n), -1)
    return r.permutation(n)


@pytest.mark.parametrize("nrhs", [1, 3, 16])
@pytest.mark.parametrize("kind", ["up", "down", "random"])
def test_exact_systems(kind, nrhs):
    systems, want = [], []
    for n in SIZES:
        r = wl.rng(100 * n + nrhs)
        i = np.arange(1, n)
        l = np.eye(n)
        l[i, i // 2] = 0.5
        u = np.diag(2.0 ** r.integers(1, 3, n))
        c = l.copy()
        for d in (1, 3, 17, 40, 130):
            if d < n:
                u += np.diag(r.integers(-2, 3, n - d).astype(float), d)
                c += np.diag(0.5 * r.integers(-1, 2, n - d), -d)
        np.fill_diagonal(c, 2.0 ** r.integers(0, 3, n))
        x = r.integers(-4, 5, (nrhs, n)).astype(float)
        p = order(kind, n, r)
        a = np.empty((n, n))
        a[p] = l @ u
        rows, ipiv = np.argsort(p), np.empty(n, dtype=np.int64)
        for k in range(n):
            ipiv[k] = q = k + int(np.flatnonzero(rows[k:] == k)[0])
            rows[[k, q]] = rows[[q, k]]
        systems += [(batch.KIND_LU, a, x @ a.T), (batch.KIND_CHOL, c @ c.T, x @ (c @ c.T))]
        want += [(x, np.tril(l, -1) + u, ipiv), (x, c, None)]
    out = batch.solve_batch(systems)
    for i, ((k, a, _), (x, f, ipiv)) in enumerate(zip(systems, want)):
        assert out["status"][i] == 0
        if ipiv is not None:
            assert np.array_equal(out["ipiv"][i], ipiv), a.shape
            assert np.array_equal(out["factor"][i], f), a.shape
        else:
            assert np.array_equal(np.tril(out["factor"][i]), f), a.shape
        assert np.array_equal(out["x"][i], x), (k, a.shape)
