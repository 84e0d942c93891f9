"""The pivot choice between workgroups of the exchange panel, on either side of 64
workgroups (16,384 rows in FP64, 32,768 in FP32: beyond that, headers are read in
rounds of 64 and rows are not read ahead).

A = P L U as in the row-step tests, exact at every step, but the first columns hold
only their pivot and one rival: of the same magnitude (the lower row wins), or
different from it only in the low word of the FP64 number (the larger wins, wherever
it is)."""
import ctypes as C

import numpy as np
import pytest

from rulinalg_amd import _lib, workloads as wl

pytestmark = pytest.mark.gpu


def rivals(n, rows):
    """(winner, loser, near): `rows` per workgroup; workgroups of the same lane and of
    other lanes of the two rounds, neighbours and the first and the last."""
    last = (n - 1) // rows
    at = lambda g, i: min(g * rows + i, n - 1)
    pairs = [(at(0, 50), at(1, 44)), (at(0, rows - 1), at(1, 0)), (at(0, 60), at(last, 20)), (at(1, 7), at(last, 30))]
    if last >= 64:
        pairs += [(at(0, 70), at(64, 9)), (at(5, 3), at(64, 10)), (at(1, 12), at(65, 1)), (at(64, 40), at(65, 40)),
                  (at(63, rows - 1), at(64, 0)), (at(2, 9), at(last, 31))]
    return [(lo, hi, False) for lo, hi in pairs[::2]] + [(hi, lo, True) for lo, hi in pairs[1::2]] + \
           [(lo + 2, hi + 2, True) for lo, hi in pairs[::2]]


@pytest.mark.parametrize("n,dt", [(600, np.float64), (16950, np.float64), (1200, np.float32), (33400, np.float32)])
def test_rivals(n, dt):
    import torch
    td, rows = (torch.float64, 256) if dt == np.float64 else (torch.float32, 512)
    r = wl.rng(n)
    special = [s for s in rivals(n, rows) if dt == np.float64 or not s[2]]
    K = len(special)
    # row k of L U is row p[k] of A
    p = np.empty(n, dtype=np.int64)
    p[:K] = [w for w, _, _ in special]
    p[K:] = r.permutation(np.setdiff1d(np.arange(n), p[:K]))
    where = np.argsort(p)
    assert len(set(p[:K]) | {s[1] for s in special}) == 2 * K and p[:K].min() >= K
    lu = torch.zeros((n, n), dtype=td, device="cuda")  # the factor, L below U
    i = torch.arange(n, device="cuda")
    lu[i, i] = torch.tensor(2.0 ** r.integers(1, 3, n), dtype=td, device="cuda")
    for d in (1, 3, 40, 70, 200):
        v = torch.tensor(r.integers(-2, 3, n - d), dtype=td, device="cuda")
        v[:K] = 0
        lu[i[:n - d], i[d:]] = v
    h = i // 2
    low = torch.where(h >= K, 0.5, 0.0).to(td)
    a = lu + low[:, None] * lu[h]
    lu[i[2 * K:], h[2 * K:]] = 0.5
    for k, (_, loser, near) in enumerate(special):
        j = int(where[loser])
        a[k, k] = lu[k, k] = 4.0 + (2.0 ** -30 if near else 0.0)
        a[j, k] = -4.0
        lu[j, k] = -4.0 / (4.0 + (2.0 ** -30 if near else 0.0))
    a[torch.tensor(p, device="cuda")] = a.clone()
    # the swaps that bring row p[k] to position k, by position and row
    row_at, at_row, ipiv = np.arange(n), np.arange(n), np.empty(n, dtype=np.int64)
    for k in range(n):
        q = ipiv[k] = at_row[p[k]]
        row_at[[k, q]] = row_at[[q, k]]
        at_row[row_at[[k, q]]] = [k, q]
    assert np.all(ipiv >= np.arange(n))
    torch.cuda.synchronize()

    lib, f = _lib.load(), C.c_void_p()
    if dt == np.float64:
        st = lib.rlg_lu_decompose_f64_dev(n, a.data_ptr(), n, None, C.byref(f))
    else:
        ah = a.cpu().numpy()
        st = lib.rlg_lu_decompose_f32(n, n, ah.ctypes.data, n, C.byref(f))
    assert st == 0, _lib.last_error()
    got = np.empty(n, dtype=np.int64)
    assert lib.rlg_lu_ipiv(f, got.ctypes.data) == 0
    if dt == np.float32:
        assert lib.rlg_lu_packed_f32(f, ah.ctypes.data, n) == 0
        a = torch.from_numpy(ah).cuda()
    assert lib.rlg_synchronize() == 0
    lib.rlg_lu_free(f)
    assert np.array_equal(got[:K], ipiv[:K]) and np.array_equal(got, ipiv)
    for k, (_, loser, near) in enumerate(special):  # a quotient that is not exact
        j = int(where[loser])
        if near:
            assert abs(float(a[j, k] - lu[j, k])) <= 2.0 ** -52
            a[j, k] = lu[j, k]
    assert torch.equal(a, lu)
