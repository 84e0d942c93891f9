"""CPU: the batched kernels' accesses to shared memory, with a poisoned gap behind
every member of its structure (tests/emu, batched_guarded).

Shared memory takes part in memory faults: a phase that is a function of its own, or
whose registers were spilled, reaches it (or scratch memory) through generic pointers,
and an access beyond its limit then faults the device (an aperture violation); only
an LDS instruction's is dropped.  Within the structure nothing faults, but an access
past one member reads or destroys another.  The orders are those at the edges of
panels, tiles and strips of tiles."""
import os
import subprocess

import numpy as np
import pytest

import test_batched_emu_cpu as emu
from rulinalg_amd import workloads as wl

pytestmark = emu.pytestmark
GUARDED = os.path.join(emu.EMU, "_build", "batched_guarded")


@pytest.fixture(scope="module", autouse=True)
def build():
    p = subprocess.run(["make", "-s", "-j4", "-C", emu.EMU], capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]


@pytest.fixture(autouse=True)
def guarded(monkeypatch):
    monkeypatch.setattr(emu, "EXE", GUARDED)


ORDERS = [1, 2, 7, 9, 15, 17, 24, 31, 33, 56, 63, 65, 120, 127, 129, 145, 247, 250, 257, 273, 385, 500, 511, 512]


@pytest.mark.parametrize("mode", [0, 1], ids=["plain", "mixed"])
@pytest.mark.parametrize("kind", [emu.LU, emu.CHOL], ids=["lu", "chol"])
def test_every_order_and_width(kind, mode):
    cases = [(n, nb) for n in ORDERS for nb in emu.widths(n)]

    def one(case):
        n, nb = case
        r = wl.rng(2000 + 7 * n + nb + kind)
        a, b = emu.system(r, kind, n, (1, 4, 16)[n % 3])
        st, fb, [(fa, x, ip)] = emu.run([(kind, a, b, nb)], mode=mode, order=n % 3, grid=2, block=1)
        return case, st, a, b, x

    for case, st, a, b, x in emu.parallel(one, cases):
        assert st == [emu.OK], case
        assert max(emu.eta(a, x[i], b[i]) for i in range(len(b))) <= 1e-13, case


def test_swaps_of_every_kind():
    """No swap, every row moved, chains through the panel: the padded list of moves."""
    systems = []
    for n, nb in ((32, 8), (64, 16), (96, 32), (150, 16), (247, 32)):
        r = wl.rng(n)
        u = np.triu(r.uniform(0.5, 1.0, (n, n))) / n + np.eye(n)
        for p in (np.arange(n), np.arange(n)[::-1], np.roll(np.arange(n), 1), np.roll(np.arange(n), -1), r.permutation(n)):
            systems.append((emu.LU, np.ascontiguousarray(u[p]), r.standard_normal((2, n)), nb))
    st, fb, out = emu.run(systems)
    assert st == [emu.OK] * len(systems)
    for (kind, a, b, nb), (fa, x, ip) in zip(systems, out):
        assert max(emu.eta(a, x[i], b[i]) for i in range(2)) <= 1e-13


def test_fallback_and_failures():
    r = wl.rng(2300)
    n = 96
    u, _ = np.linalg.qr(r.standard_normal((n, n)))
    v, _ = np.linalg.qr(r.standard_normal((n, n)))
    sing, indef = r.standard_normal((64, 64)), np.eye(48)
    sing[:, 10], indef[20, 20] = 0.0, -1.0
    systems = [(emu.LU, (u * np.logspace(0, -9, n)) @ v.T, r.standard_normal((2, n)), 16),
               (emu.LU, sing, r.standard_normal((1, 64)), 8), (emu.CHOL, indef, r.standard_normal((1, 48)), 16)]
    want = [emu.OK, emu.DIV_BY_ZERO, emu.DECOMP_FAILURE]
    assert emu.run(systems, mode=1, grid=4, block=3)[0] == want
    assert emu.run(systems)[0] == want


def test_a_planted_access_is_reported():
    p = subprocess.run([emu.SELFTEST, "gap", "0"], capture_output=True, text=True, timeout=60, env=emu.ENV)
    assert p.returncode != 0 and "use-after-poison" in p.stderr, p.stderr[-2000:]
