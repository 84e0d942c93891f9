"""Products so tall that narrow tiles would need more threads than one launch can
have (2^32).  One term per entry, so every entry is exact."""
import pytest

from rulinalg_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m", [2 ** 29, 2 ** 30 - 1])
def test_tall(m, trans):
    import torch
    lib = _lib.load()
    a = (torch.arange(m, device="cuda", dtype=torch.int32) & 0xFFFF).to(torch.float32)
    b = torch.full((1,), 3.0, device="cuda")
    c = torch.zeros_like(a)
    torch.cuda.synchronize()
    if trans:  # a row of that length
        assert lib.rlg_gemm_f32_dev(1, 1, m, 1.0, b.data_ptr(), 1, a.data_ptr(), m, 0.0, c.data_ptr(), m, None) == 0, \
            _lib.last_error()
    else:
        assert lib.rlg_gemm_f32_dev(m, 1, 1, 1.0, a.data_ptr(), 1, b.data_ptr(), 1, 0.0, c.data_ptr(), 1, None) == 0, \
            _lib.last_error()
    assert lib.rlg_synchronize() == 0
    a *= 3.0
    assert torch.equal(a, c)
