"""17 .. 32 token columns: the streaming kernel's tiles of 32 tokens give the bits of its tiles of 64 (a column's sums do not depend on the tile), for every
height of its row tiles, whole and in K slices, on both sides of the tile's edges and of K shorter than its rings; and both stay at the product."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, k: 24-, 40-, 48-, 56-, 80- and 96-row tiles with a last one cut short, then K slices (80-, 16- and 64-row tiles; 8 k tiles a slice, 19, 5, 4)
SHAPES = [(6144, 2560), (4108, 64), (4100, 1088), (10236, 640), (11244, 640), (14004, 2560), (19452, 192), (24000, 1088), (2560, 4096), (2556, 9728), (512, 2560), (2048, 2048)]


def _draw(*shape, seed):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed))


@pytest.mark.parametrize("M,K", SHAPES)
@pytest.mark.parametrize("gated", [False, True])
def test_columns(M, K, gated):
    from pegainfer_amd import ops as P
    W, X = (_draw(M, K, seed=M + K) / K ** 0.5).bfloat16(), _draw(64, K, seed=K).bfloat16()

    def run(T):
        out = torch.full((T + 1, M // 2 if gated else M), 9.0, device="cuda", dtype=torch.bfloat16)
        (P.gemm_silu_into if gated else P.gemm_into)(W, X[:T], out[:T])
        assert bool((out[T] == 9).all())
        return out[:T]
    ref = X.float() @ W.float().T
    if gated:
        g, u = ref.bfloat16().float().chunk(2, 1)
        ref = g * torch.sigmoid(g) * u
    whole = run(64)
    # a sum of K products in fp32 and up to three roundings to bf16, of the gate and up values and the result: 2^-9 each, the gate's twice over
    assert float((whole.float() - ref).norm() / ref.norm()) < 4 * 2 ** -8
    for T in (17, 31, 32, 33):
        assert torch.equal(run(T), whole[:T]), T
