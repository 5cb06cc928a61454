"""The clamped gated unit in its projections' launch against the product and the unit one after the other: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("I,K", [(1, 8), (7, 504), (300, 1000), (1024, 2560), (513, 4096), (66, 9216), (96, 20000)])
def test_as_two_launches(T, I, K):
    from pegainfer_amd import ffi, ops_blocks as B
    L, s = ffi.lib(), B._stream()
    g = torch.Generator().manual_seed(I + K)
    w, x = (torch.randn(*sh, generator=g).bfloat16().cuda() for sh in ((2 * I, K), (T, K)))
    w *= 8 * K ** -0.5                                   # values on both sides of the limit
    gu, a, b = (torch.zeros(T, n, dtype=torch.bfloat16, device="cuda") for n in (2 * I, I, I))
    L.gemm_cuda(w.data_ptr(), x.data_ptr(), gu.data_ptr(), 2 * I, T, K, s)
    assert L.pegainfer_clamp_glu_rows(gu.data_ptr(), a.data_ptr(), I, T, 7.0, 1.702, 0, s) == 0
    assert L.pegainfer_gemv_clamp_glu_ok(w.data_ptr(), x.data_ptr(), T, K)
    assert L.pegainfer_gemv_clamp_glu(w.data_ptr(), x.data_ptr(), b.data_ptr(), I, T, K, 7.0, 1.702, s) == 0
    assert torch.equal(a, b) and torch.isfinite(a.float()).all() and float(a.float().abs().max()) > 0


def test_what_it_leaves_to_two_launches():
    from pegainfer_amd import ffi
    x = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda")
    ok = lambda T, K, at=0: ffi.lib().pegainfer_gemv_clamp_glu_ok(x.data_ptr() + at, x.data_ptr(), T, K)
    assert ok(1, 64) and not ok(3, 64) and not ok(1, 60) and not ok(1, 64, 2)
