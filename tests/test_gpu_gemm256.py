"""The 256 x 256 GEMM at the edges of its tiles and of its ways out (whole rows of 16 bytes, halves of 8, value by value): against the product in
double precision, within the bf16 rounding of the result and a sum of K products of about one in fp32 (1e-6 K, four times that for the order)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _route(M, T, K, I=0):
    from pegainfer_amd import ffi
    out = (ctypes.c_int32 * 3)()
    assert ffi.lib().pegainfer_debug_gemm_route(M, T, K, I, out) == 0
    return out[0]


def _operands(M, T, K):
    g = torch.Generator(device="cuda").manual_seed(M + T + K)
    return torch.randn(M, K, device="cuda", generator=g).bfloat16(), torch.randn(T, K, device="cuda", generator=g).bfloat16()


def _close(Y, ref, K):
    return bool(((Y.double() - ref).abs() <= 4e-6 * K + ref.abs() * 2.0 ** -8).all())


# two K tile pairs and more, a row or a token more than whole tiles, rows that end inside a chunk of eight and of four; more tiles than workgroups
@pytest.mark.parametrize("M,T,K", [(32768, 256, 256), (32768, 257, 384), (16385 + 255, 513, 256), (8193 + 511, 1023, 512), (16396, 511, 256), (5128, 2049, 640),
                                   (5124, 2305, 256), (12800, 2049, 384), (12804, 2100, 256), (2560, 9990, 768)])
def test_plain(M, T, K):
    from pegainfer_amd import ops as P
    assert _route(M, T, K) in (256, 259)
    W, X = _operands(M, T, K)
    Y = torch.full((T, M), float("nan"), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, Y)
    assert _close(Y, X.double() @ W.double().T, K)


# segments on whole chunks of eight, and inside a chunk (4 mod 8): the most that the entry point hands to these tiles
@pytest.mark.parametrize("parts", [(4096, 1024, 1024), (4100, 1020, 1024), (4100, 1020, 1028), (8, 6128, 8), (4, 6136, 4)])
def test_segments(parts):
    from pegainfer_amd import ops as P
    M, T, K = sum(parts), 1600, 256
    assert _route(M, T, K) == 256 and all(m % 4 == 0 for m in parts)
    W, X = _operands(M, T, K)
    ys = [torch.full((T, m), float("nan"), device="cuda", dtype=torch.bfloat16) for m in parts]
    P.gemm_split3_into(W, X, *ys)
    assert _close(torch.cat(ys, 1), X.double() @ W.double().T, K)


def test_segments_that_are_no_fours_run_as_products_of_their_own():
    from pegainfer_amd import ops as P
    parts, T, K = (4097, 1021, 1026), 1600, 256
    W, X = _operands(sum(parts), T, K)
    ys = [torch.full((T, m), float("nan"), device="cuda", dtype=torch.bfloat16) for m in parts]
    P.gemm_split3_into(W, X, *ys)
    assert _close(torch.cat(ys, 1), X.double() @ W.double().T, K)


@pytest.mark.parametrize("M,T,K", [(2560, 2047, 4096), (2568, 1500, 4224), (2562, 1793, 4096), (2048, 1536, 4224)])
def test_slices_of_k(M, T, K):
    from pegainfer_amd import ops as P
    assert _route(M, T, K) == 1256
    W, X = _operands(M, T, K)
    Y = torch.full((T, M), float("nan"), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, Y)
    assert _close(Y, X.double() @ W.double().T, K)


@pytest.mark.parametrize("I,T,K", [(16384, 256, 256), (9224, 600, 256), (9220, 513, 256), (9219, 512, 384), (12808, 1000, 256), (12801, 1000, 256)])
def test_gated_unit_has_the_bits_of_product_and_unit(I, T, K):
    from pegainfer_amd import ops as P
    assert _route(0, T, K, I) in (256, 257)
    W, X = _operands(2 * I, T, K)
    W *= 0.3
    fused = torch.full((T, I), float("nan"), device="cuda", dtype=torch.bfloat16)
    P.gemm_silu_into(W, X, fused)
    both = torch.empty((T, 2 * I), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, both)
    two = torch.empty((T, I), device="cuda", dtype=torch.bfloat16)
    P.silu_mul_fused_batch_into(both, two)
    assert torch.equal(fused, two)


def test_gated_unit_over_every_finite_gate():
    """a row of weights per bf16 pattern, its only value beside zeros: the gate is that value exactly.  Bits, the sign of zero among them."""
    from pegainfer_amd import ops as P
    I, T, K = 65536 - 512, 256, 256
    bits = torch.arange(65536, device="cuda", dtype=torch.int32)
    bits = bits[(bits & 0x7F80) != 0x7F80]                       # finite ones
    gate = bits[:I].to(torch.int16).view(torch.bfloat16)
    assert gate.numel() == I and _route(0, T, K, I) == 256
    W = torch.zeros(2 * I, K, device="cuda", dtype=torch.bfloat16)
    W[:I, 3] = gate
    W[I:, 5] = 1.0
    X = torch.zeros(T, K, device="cuda", dtype=torch.bfloat16)
    X[:, 3] = 1.0
    X[:, 5] = torch.linspace(-3, 3, T, device="cuda").bfloat16()
    fused = torch.empty((T, I), device="cuda", dtype=torch.bfloat16)
    P.gemm_silu_into(W, X, fused)
    both = torch.empty((T, 2 * I), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, both)
    two = torch.empty((T, I), device="cuda", dtype=torch.bfloat16)
    P.silu_mul_fused_batch_into(both, two)
    assert torch.equal(both[0, :I].view(torch.int16)[gate.view(torch.int16) != -32768], gate.view(torch.int16)[gate.view(torch.int16) != -32768])
    assert torch.equal(fused.view(torch.int16), two.view(torch.int16))
