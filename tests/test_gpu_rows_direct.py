"""Up to four fp32 rows against fp32 weights, and one fp32 row against bf16 weights, without LDS: pieces of k that end inside a wave's 512, outputs past a
wave's last, groups, gathered and scattered rows, a table's tiles, and pairs of rows under a gated unit.  Against double precision; a sum of K
products of about one in fp32: 1e-6 K."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 3, 4])
@pytest.mark.parametrize("M,K", [(1, 8), (7, 520), (1024, 512), (1025, 1000), (2051, 1544), (4099, 1032), (9000, 2056)])
def test_few_fp32_rows(T, M, K):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator(device="cuda").manual_seed(T * 1000 + M + K)
    x = torch.full((T + 3, K + 8), float("nan"), device="cuda")          # what lies behind a row is never used
    w = torch.full((2, M, K + 8), float("nan"), device="cuda")
    x[:, :K], w[..., :K] = torch.randn(T + 3, K, device="cuda", generator=g), torch.randn(2, M, K, device="cuda", generator=g)
    y = torch.full((T + 2, 2 * M), float("nan"), device="cuda")
    src = torch.randperm(T + 3, device="cuda", generator=g)[:T].int()
    dst = torch.randperm(T + 2, device="cuda", generator=g)[:T].int()
    B.gemm_strided(B.GemmDesc(x=x.data_ptr(), w=w.data_ptr(), y=y.data_ptr(), x_dtype=1, w_dtype=1, y_dtype=1, m=M, k=K, rows=T, groups=2,
                              x_row_stride=K + 8, w_m_stride=K + 8, w_k_stride=1, w_group_stride=M * (K + 8), y_row_stride=2 * M, y_group_stride=M,
                              x_row_index=src.data_ptr(), y_row_index=dst.data_ptr(), epilogue=B.EPI_RELU_SQ))
    ref = torch.relu(torch.einsum("tk,gmk->tgm", x[src.long(), :K].double(), w[..., :K].double())) ** 2
    got = y[dst.long()].view(T, 2, M).double()
    assert float((got - ref).abs().max()) <= 1e-6 * K * (1 + float(ref.sqrt().max()))
    left = torch.ones(T + 2, dtype=torch.bool, device="cuda")
    left[dst.long()] = False
    assert bool(y[left].isnan().all())
    if T == 1:                                                           # one fp32 row against bf16 weights, and what a row gives alone and beside others
        wb = torch.zeros(M, K + 8, device="cuda", dtype=torch.bfloat16)
        wb[:, :K] = w[0, :, :K]
        yb = torch.empty(1, M, device="cuda")
        B.gemm_strided(B.GemmDesc(x=x.data_ptr(), w=wb.data_ptr(), y=yb.data_ptr(), x_dtype=1, w_dtype=0, y_dtype=1, m=M, k=K, rows=1, groups=1,
                                  x_row_stride=K + 8, w_m_stride=K + 8, w_k_stride=1, y_row_stride=M))
        assert float((yb[0].double() - wb[:, :K].double() @ x[0, :K].double()).abs().max()) <= 1e-6 * K


@pytest.mark.parametrize("act", [0, 1, 2, 3])
@pytest.mark.parametrize("T,M,K", [(1, 5, 72), (2, 3072, 1024), (3, 1030, 520), (4, 513, 1544)])
def test_gated_unit_of_few_fp32_rows(act, T, M, K):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator(device="cuda").manual_seed(act * 10 + T + M)
    x, w = torch.randn(T, K, device="cuda", generator=g), torch.randn(2 * M + 3, K, device="cuda", generator=g) / K ** 0.5
    y = torch.full((T, M), float("nan"), device="cuda")
    B.glu_gemm(B.GluGemmDesc(g=B.GemmDesc(x=x.data_ptr(), w=w.data_ptr(), y=y.data_ptr(), x_dtype=1, w_dtype=1, y_dtype=1, m=M, k=K, rows=T, groups=1,
                                          x_row_stride=K, w_m_stride=K, w_k_stride=1, y_row_stride=M), act=act, up=(M + 3) * K))
    z = x.double() @ w.double().T
    a, u = z[:, :M], z[:, M + 3:]
    f = [lambda t: t * torch.sigmoid(t), torch.relu, lambda t: torch.nn.functional.gelu(t, approximate="tanh"), torch.nn.functional.gelu][act]
    # a pair's sums are off by 1e-6 sqrt(K) each, the activation's slope is about one and fp32 functions add a few ulp
    assert float((y.double() - f(a) * u).abs().max()) <= 1e-6 * (K ** 0.5 + 8) * float(1 + z.abs().max()) * 2


@pytest.mark.parametrize("wd,T", [(torch.float32, 1), (torch.float32, 2), (torch.float32, 4), (torch.bfloat16, 1)])
@pytest.mark.parametrize("M,K", [(3200, 264), (5000, 512), (9000, 1040), (8500, 4104), (4200, 2056)])
def test_an_output_does_not_depend_on_how_many_a_wave_makes(wd, T, M, K):
    """one, two or four outputs a wave by their number, the row's length and the rows: the bits of a launch of a few (one a wave), and double precision"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator(device="cuda").manual_seed(M + T)
    x, w = torch.randn(T, K, device="cuda", generator=g), torch.randn(M, K, device="cuda", generator=g).to(wd)
    y = B.linear(x, w, out_dtype=torch.float32)
    for at in (0, M // 2, M - 77):
        assert torch.equal(y[:, at:at + 77], B.linear(x, w[at:at + 77].contiguous(), out_dtype=torch.float32)), at
    assert float((y.double() - x.double() @ w.double().T).abs().max()) <= 1e-6 * K


def test_other_gated_units_are_refused():
    from pegainfer_amd import ops_blocks as B
    x, w, y = torch.zeros(5, 64, device="cuda"), torch.zeros(16, 64, device="cuda"), torch.zeros(5, 8, device="cuda")
    d = dict(x=x.data_ptr(), w=w.data_ptr(), y=y.data_ptr(), x_dtype=1, w_dtype=1, y_dtype=1, m=8, k=64, rows=2, groups=1, x_row_stride=64, w_m_stride=64,
             w_k_stride=1, y_row_stride=8)
    for change, more in ((dict(rows=5), {}), (dict(k=60), {}), (dict(epilogue=B.EPI_RELU_SQ), {}), ({}, dict(up=4)), ({}, dict(act=4))):
        with pytest.raises(RuntimeError):
            B.glu_gemm(B.GluGemmDesc(g=B.GemmDesc(**{**d, **change}), **{**dict(act=0, up=8 * 64), **more}))
