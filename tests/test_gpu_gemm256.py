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


@pytest.mark.parametrize("M,T,K", [(2560, 2047, 4096), (2568, 1500, 4224), (2564, 1793, 4096), (2048, 1536, 4224)])
def test_slices_of_k(M, T, K):
    from pegainfer_amd import ops as P
    assert _route(M, T, K) == 1256 and M % 4 == 0
    W, X = _operands(M, T, K)
    Y = torch.full((T, M), float("nan"), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, Y)
    assert _close(Y, X.double() @ W.double().T, K)


def _unit(both, rounded):
    """the gated unit behind the product, in a launch of its own"""
    from pegainfer_amd import ops as P
    I = both.shape[1] // 2
    two = torch.empty((both.shape[0], I), device="cuda", dtype=torch.bfloat16)
    if rounded:
        P.silu_mul_batch_into(both[:, :I].contiguous(), both[:, I:].contiguous(), two)
    else:
        P.silu_mul_fused_batch_into(both, two)
    return two


def _fused(W, X, rounded):
    from pegainfer_amd import ffi
    I, (T, K) = W.shape[0] // 2, X.shape
    Y = torch.full((T, I), float("nan"), device="cuda", dtype=torch.bfloat16)
    scratch = torch.empty((T, 2 * I), device="cuda", dtype=torch.bfloat16)
    f = ffi.lib().pegainfer_gemm_silu_rounded if rounded else ffi.lib().pegainfer_gemm_silu
    assert f(W.data_ptr(), X.data_ptr(), Y.data_ptr(), scratch.data_ptr(), I, T, K, torch.cuda.current_stream().cuda_stream) == 0
    return Y


# (columns that are not multiples of four never come to these tiles: the two launches run instead)
@pytest.mark.parametrize("rounded", [False, True])
@pytest.mark.parametrize("I,T,K", [(16384, 256, 256), (9224, 600, 256), (9220, 513, 256), (10244, 512, 384), (12808, 1000, 256), (12804, 1000, 256)])
def test_gated_unit_has_the_bits_of_product_and_unit(I, T, K, rounded):
    from pegainfer_amd import ops as P
    assert _route(0, T, K, I) in (256, 257) and I % 4 == 0
    W, X = _operands(2 * I, T, K)
    W *= 0.3
    both = torch.empty((T, 2 * I), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, both)
    assert torch.equal(_fused(W, X, rounded), _unit(both, rounded))


@pytest.mark.parametrize("rounded", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
def test_gated_unit_over_every_finite_gate(mixed, rounded):
    """a row of weights per finite bf16 pattern, its only value beside zeros: the gate is that value exactly.  A wave takes the short form of the unit where
    all of its 64 columns' gates have 0 < |g| <= 80: those stand together, 64 and 64, and the others behind them; mixed, every wave meets both kinds.
    Bits, the sign of zero among them."""
    from pegainfer_amd import ops as P
    size = torch.arange(0x7F80, dtype=torch.int32)
    short = size[(size > 0) & (size <= 0x42A0)]
    other = size[(size == 0) | (size > 0x42A0)]
    pad = lambda v, with_: torch.cat([v, torch.full((-len(v) % 64,), with_, dtype=v.dtype)])   # noqa: E731
    order = torch.cat([pad(torch.cat([short, short | 0x8000]), 0x3F80), pad(torch.cat([other, other | 0x8000]), 0x7F00)])
    assert len(set(order.tolist())) == 2 * 0x7F80
    if mixed:
        order = order[torch.randperm(len(order), generator=torch.Generator().manual_seed(3))]
    gate = order.to(torch.int16).view(torch.bfloat16).cuda()
    I, T, K = len(order), 256, 256
    assert I % 128 == 0 and _route(0, T, K, I) == 256            # whole tiles: a wave's columns begin on 64
    W = torch.zeros(2 * I, K, device="cuda", dtype=torch.bfloat16)
    W[:I, 3] = gate
    W[I:, 5] = 1.0
    X = torch.zeros(T, K, device="cuda", dtype=torch.bfloat16)
    X[:, 3] = 1.0
    X[:, 5] = torch.linspace(-3, 3, T, device="cuda").bfloat16()
    both = torch.empty((T, 2 * I), device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, both)
    got = both[0, :I].view(torch.int16)
    assert bool(((got == gate.view(torch.int16)) | (gate == 0)).all())
    assert torch.equal(_fused(W, X, rounded).view(torch.int16), _unit(both, rounded).view(torch.int16))
