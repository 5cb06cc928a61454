"""Few normed rows of more than 2560 values in front of a product: the bits of the norm and the product as launches of their own, at both ends of the
range of lengths and of rows a wave stages."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [3, 8, 9, 16])
@pytest.mark.parametrize("K", [2560, 2688, 3968, 4096, 4224])
@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("gated", [False, True])
def test_norm_in_front_of_few_rows(T, K, residual, gated):
    from pegainfer_amd import ffi
    from pegainfer_amd import ops as P
    g = torch.Generator(device="cuda").manual_seed(T * K)
    M = 1300
    W = (torch.randn(M, K, device="cuda", generator=g) * 0.05).bfloat16()
    X, R = (torch.randn(T, K, device="cuda", generator=g).bfloat16() for _ in "xr")
    gain = (1 + 0.2 * torch.randn(K, device="cuda", generator=g)).bfloat16()
    hidden, normed, left = X.clone(), torch.empty_like(X), torch.full_like(X, 9)
    if residual:
        P.fused_add_rms_norm_batch_into(hidden, R, gain, 1e-6, normed)
    else:
        P.rms_norm_batch_into(X, gain, 1e-6, normed)
    ref = P.gemm(W, normed)
    if gated:
        both, ref = ref, torch.empty(T, M // 2, device="cuda", dtype=torch.bfloat16)
        P.silu_mul_fused_batch_into(both, ref)
    out = torch.full_like(ref, float("nan"))
    s = torch.cuda.current_stream().cuda_stream
    assert ffi.lib().pegainfer_gemv_fused(W.data_ptr(), X.data_ptr(), out.data_ptr(), M, T, K, R.data_ptr() if residual else None, gain.data_ptr(),
                                          left.data_ptr() if residual else None, 1e-6, M // 2 if gated else 0, s) == 0
    assert torch.equal(out, ref)
    if residual:
        assert torch.equal(left, hidden)
