"""Tournament panels at the edges of their tile (256 rows, groups of 16 columns,
merges of four) and with swaps that chain through the panel's top rows.

A = P (4 I + E) with |E| small: well conditioned (condition number below 3), so
that FP32 factors must refine to FP64 accuracy without a fallback, and pivot j is
the row that P puts there."""
import numpy as np
import pytest

import rulinalg_amd as rl
from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu
TOL = 1e-13  # the refinement stops at its default tolerance on the normwise backward error


def eta(a, x, b):
    return np.abs(b - a @ x).max() / (np.abs(a).sum(1).max() * np.abs(x).max() + np.abs(b).max())


def order(kind, n, r):
    if kind == "up":        # row 0 is moved on by every step
        return np.roll(np.arange(n), 1)
    if kind == "down":
        return np.roll(np.arange(n), -1)
    if kind == "reversed":
        return np.arange(n)[::-1].copy()
    return r.permutation(n)


@pytest.mark.parametrize("kind", ["up", "down", "reversed", "random"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 80, 255, 256, 257, 320, 1024, 1025])
def test_panel_edges(n, kind):
    r = wl.rng(n)
    a = 4.0 * np.eye(n) + r.uniform(-1, 1, (n, n)) / n
    a = a[order(kind, n, r)]
    b = wl.gaussian(2, n, 3)
    x, rep = rl.solve_mixed(a, b, rl.MixedOptions(factor_prec=_lib.PREC_F32, pivot=_lib.PIVOT_TOURNAMENT))
    assert rep["converged"] == 1 and rep["fell_back"] == 0
    # FP32 factors with |E| <= 1 leave at most 4 n 2^-24 of the residual per step
    assert rep["iterations"] <= 6
    for i in range(2):
        assert eta(a, x[i], b[i]) <= TOL


@pytest.mark.parametrize("n", [64, 257, 600])
def test_ties_and_zeros(n):
    """Equal candidates in every column, and columns that are zero in most leaves."""
    r = wl.rng(n)
    a = r.choice([-1.0, 1.0], (n, n))
    a[n // 2:, : n // 4] = 0.0
    a += n * np.eye(n)[r.permutation(n)]
    b = wl.gaussian(1, n, 4)
    x, rep = rl.solve_mixed(a, b, rl.MixedOptions(factor_prec=_lib.PREC_F32, pivot=_lib.PIVOT_TOURNAMENT))
    assert rep["converged"] == 1 and rep["fell_back"] == 0
    assert eta(a, x[0], b[0]) <= TOL
