"""17 .. 32 token columns: the streaming kernel's tiles of 32 tokens give the bits of its tiles of 64 (a column's sums do not depend on the tile), for every
height of its row tiles, whole and in K slices, on both sides of the tile's edges and of K shorter than its rings; and both stay at the product."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, k: 24-, 40-, 48-, 56-, 80- and 96-row tiles with a last one cut short, then K slices (80-, 16- and 64-row tiles; 8 k tiles a slice, 19, 5, 4)
SHAPES = [(6144, 2560), (4108, 64), (4100, 1088), (10236, 640), (11244, 640), (14004, 2560), (19452, 192), (24000, 1088), (2560, 4096), (2556, 9728), (512, 2560), (2048, 2048)]
# gated columns, k, 16-row blocks of the tile: 12, 20 and 40 columns and their up rows, the last tile cut short, K shorter than the rings and not
GATED = [(2056, 64, 2), (2056, 1088, 2), (5116, 128, 4), (5116, 640, 4), (5116, 1088, 4), (9724, 192, 6), (9724, 1088, 6), (9724, 2560, 6)]


def _draw(*shape, seed):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed))


def _route(M, T, K, I=0):
    from pegainfer_amd import ffi
    out = (ctypes.c_int32 * 3)()
    assert ffi.lib().pegainfer_debug_gemm_route(M, T, K, I, out) == 0
    return out[0]


@pytest.mark.parametrize("M,K", SHAPES)
def test_columns(M, K):
    from pegainfer_amd import ops as P
    W, X = (_draw(M, K, seed=M + K) / K ** 0.5).bfloat16(), _draw(64, K, seed=K).bfloat16()

    def run(T):
        assert _route(M, T, K) // 1000 in (2, 3) and M % 4 == 0
        out = torch.full((T + 1, M), 9.0, device="cuda", dtype=torch.bfloat16)
        P.gemm_into(W, X[:T], out[:T])
        assert bool((out[T] == 9).all())
        return out[:T]
    ref = X.float() @ W.float().T
    whole = run(64)
    # a sum of K products in fp32 and a rounding to bf16, 2^-9
    assert float((whole.float() - ref).norm() / ref.norm()) < 2 ** -8
    for T in (17, 31, 32, 33):
        assert torch.equal(run(T), whole[:T]), T


# (2058 columns, no multiple of four, and 1280, whose product runs in K slices, take the product and the unit in launches of their own)
@pytest.mark.parametrize("I,K,blocks", GATED + [(2058, 640, 0), (1280, 4096, 0)])
def test_gated_columns(I, K, blocks):
    from pegainfer_amd import ops as P
    W, X = (_draw(2 * I, K, seed=I + K) / K ** 0.5).bfloat16(), _draw(64, K, seed=K).bfloat16()

    def run(T):
        if blocks:
            assert _route(0, T, K, I) == 3000 + blocks and _route(2 * I, T, K) > 3000 and I % 4 == 0
        out = torch.full((T + 1, I), 9.0, device="cuda", dtype=torch.bfloat16)
        P.gemm_silu_into(W, X[:T], out[:T])
        assert bool((out[T] == 9).all())
        return out[:T]
    both, two = torch.empty(64, 2 * I, device="cuda", dtype=torch.bfloat16), torch.empty(64, I, device="cuda", dtype=torch.bfloat16)
    P.gemm_into(W, X, both)
    P.silu_mul_fused_batch_into(both, two)
    for T in (17, 31, 32, 33, 64):
        assert torch.equal(run(T), two[:T]), T
    g, u = (X.float() @ W.float().T).bfloat16().float().chunk(2, 1)
    ref = g * torch.sigmoid(g) * u
    # up to three roundings to bf16, of the gate and up values and the result: 2^-9 each, the gate's twice over
    assert float((two.float() - ref).norm() / ref.norm()) < 4 * 2 ** -8
