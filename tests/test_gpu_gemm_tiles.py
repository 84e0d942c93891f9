"""The product's tile edges (32, 64, 128), its 16-byte and scalar tile loads and
its shallow (k <= 64) form, at sizes one off each tile and stage boundary.

Bound: |C - C_ref| <= (k + 2) u |alpha| |A||B| + 2 u |beta C| elementwise for any
order of summation, with C_ref in FP64 (its own error, k 2^-53 |A||B|, is added
for FP64 operands)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _product(torch, lib, m, k, n, pad, dt, alpha, beta):
    g = torch.Generator(device="cuda").manual_seed(m * 7 + k * 3 + n)
    a = torch.rand(m, k + pad, dtype=dt, device="cuda", generator=g) - 0.5
    b = torch.rand(k, n + pad, dtype=dt, device="cuda", generator=g) - 0.5
    c = torch.rand(m, n + pad, dtype=dt, device="cuda", generator=g) - 0.5
    c0 = c.clone()
    torch.cuda.synchronize()
    f = lib.rlg_gemm_f64_dev if dt == torch.float64 else lib.rlg_gemm_f32_dev
    assert f(m, k, n, alpha, a.data_ptr(), k + pad, b.data_ptr(), n + pad, beta, c.data_ptr(), n + pad, None) == 0
    assert lib.rlg_synchronize() == 0
    ad, bd, cd = (t.cpu().numpy().astype(np.float64) for t in (a[:, :k], b[:, :n], c0[:, :n]))
    u = 2.0 ** -53 if dt == torch.float64 else 2.0 ** -24
    ref = alpha * (ad @ bd) + beta * cd
    mag = abs(alpha) * (np.abs(ad) @ np.abs(bd))
    bound = (k + 2) * u * mag + 2 * u * np.abs(beta * cd) + u * np.abs(ref) + k * 2.0 ** -53 * mag
    assert np.all(np.abs(c[:, :n].cpu().numpy().astype(np.float64) - ref) <= bound)
    if pad:  # nothing is written past the columns
        assert torch.equal(c[:, n:], c0[:, n:])


@pytest.mark.parametrize("dt", ["float64", "float32"])
@pytest.mark.parametrize("m,k,n,pad", [
    (31, 16, 33, 0), (32, 65, 32, 0), (33, 129, 31, 1),        # 32-wide tiles
    (1000, 96, 1023, 1), (1056, 80, 1024, 0),                  # 64-wide tiles
    (2049, 97, 2047, 0), (2052, 100, 2044, 0),                 # 128-wide tiles, both loads
    (2049, 63, 2047, 0), (130, 64, 132, 0), (65, 1, 63, 1),    # shallow
])
def test_tile_edges(dt, m, k, n, pad):
    torch = pytest.importorskip("torch")
    from rulinalg_amd import _lib
    lib = _lib.load()
    for alpha, beta in ((1.0, 0.0), (-1.0, 1.0), (0.5, -2.0)):
        _product(torch, lib, m, k, n, pad, getattr(torch, dt), alpha, beta)
