"""Plain GEMMs whose rows behind the full rounds of 256 x 256 tiles run on smaller tiles: the same bits as the same rows inside the full rounds
have, the full rounds the bits of a launch without the others, and the double-precision product within a sum of K products of about one in fp32 (1e-6 K) and the bf16 rounding of the result."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,T,K,kernel", [(16392, 1024, 256, 64), (16900, 1000, 384, 64), (8192, 2057, 256, 64), (19476, 1024, 256, 96),
                                          (8448, 2404, 256, 96)])
@pytest.mark.parametrize("outputs", [1, 3])
def test_rows_behind_the_full_rounds(M, T, K, kernel, outputs):
    from pegainfer_amd import ffi
    from pegainfer_amd import ops as P
    out = (ctypes.c_int32 * 2)()
    assert ffi.lib().pegainfer_debug_gemm_tail(M, T, K, out) == 0 and out[1] == kernel
    cut = out[0] * 256
    assert 0 < cut < M
    g = torch.Generator(device="cuda").manual_seed(M + T)
    W = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    X = torch.randn(T, K, device="cuda", generator=g).bfloat16()
    if outputs == 1:
        Y = torch.full((T, M), float("nan"), device="cuda", dtype=torch.bfloat16)
        P.gemm_into(W, X, Y)
    else:                                       # cut apart on both sides of the hand-off
        a, b = cut - 128, 132
        ys = [torch.full((T, m), float("nan"), device="cuda", dtype=torch.bfloat16) for m in (a, b, M - a - b)]
        P.gemm_split3_into(W, X, *ys)
        Y = torch.cat(ys, 1)
    head = torch.empty((T, cut), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W[:cut], X, head)
    assert torch.equal(Y[:, :cut], head)
    rolled = torch.empty((T, M), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W.roll(M - cut, 0), X, rolled)   # the rows behind the cut come first: in the full rounds
    assert torch.equal(Y[:, cut:], rolled[:, :M - cut])
    ref = X.double() @ W.double().T
    tol = 1e-6 * K * 4 + ref.abs() * 2.0 ** -8
    assert bool(((Y.double() - ref).abs() <= tol).all())
