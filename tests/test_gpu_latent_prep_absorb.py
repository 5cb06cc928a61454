"""The prep of a latent attention and the product that carries its queries into the latent space in one launch: the same bits as the two launches,
at row counts around the forms' edges, with and without each part of the prep; and what the launch does not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def parts(dtype, T, H, dn, dr, r, seed=0):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(seed + T * 7 + r)
    draw = lambda *s: torch.randn(*s, generator=g).to(DT[dtype]).cuda()
    E, qr, ps = r + dr, 40, 16
    starts = [int(t) for t in torch.randint(0, 100, (T,), generator=g)]
    pages = [-(-(t + 1) // ps) for t in starts]
    indptr = torch.tensor([sum(pages[:i]) for i in range(T + 1)], dtype=torch.int32).cuda()
    pids = torch.randperm(sum(pages), generator=g).to(torch.int32).cuda()
    rg = B.Ragged([1] * T, starts=starts)
    width = -(-(H * (dn + dr) + E + qr) // 8) * 8
    proj, uk = draw(T, width), draw(H, r, dn)
    f = torch.tensor([100.0 ** (-2.0 * i / dr) for i in range(dr // 2)], dtype=torch.float32).cuda()
    norm, qnorm = draw(r), draw(qr)

    def run(together, full):
        cache = torch.zeros(sum(pages), ps * E, dtype=DT[dtype], device="cuda")
        qc = torch.full((T, H, E), float("nan"), dtype=torch.float32, device="cuda")
        d = B.GemmDesc(x=proj.data_ptr(), w=uk.data_ptr(), y=qc.data_ptr(), x_dtype=B._dt(proj), w_dtype=B._dt(uk), y_dtype=1, m=r, k=dn, rows=T,
                       groups=H, x_row_stride=width, x_group_stride=dn + dr, w_m_stride=dn, w_k_stride=1, w_group_stride=dn * r, y_row_stride=H * E,
                       y_group_stride=E)
        kw = dict(dkv=proj[:, H * (dn + dr):], c_norm_w=norm, ql=proj[:, H * (dn + dr) + E:][:, :qr], ql_norm_w=qnorm) if full else {}
        ql = B.latent_prep_form(rg, indptr, pids, cache, ps * E, 0, ps, H, dn, dr, r, 1e-5, f, not full, q=proj, qc=qc, absorb=d if together else None,
                                **kw)
        if not together:
            B.gemm_strided(d)
        return ql, qc, cache

    return run


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("dtype,T,H,dn,dr,r", [("bfloat16", 1, 3, 8, 8, 24), ("bfloat16", 16, 2, 72, 16, 40), ("bfloat16", 5, 16, 128, 64, 512),
                                               ("bfloat16", 16, 64, 64, 32, 272), ("float32", 1, 2, 8, 8, 16), ("float32", 2, 8, 64, 32, 256),
                                               ("float32", 3, 5, 40, 24, 68), ("float32", 4, 8, 128, 64, 256)])
def test_both_as_by_themselves(dtype, T, H, dn, dr, r, full):
    run = parts(dtype, T, H, dn, dr, r)
    for a, b in zip(run(False, full), run(True, full)):
        assert (a is None and b is None) or torch.equal(a, b)
    assert torch.isfinite(run(True, full)[1]).all()


def test_what_the_launch_leaves_to_two():
    assert parts("bfloat16", 17, 2, 64, 16, 32)(True, True)[0] is False
    assert parts("float32", 5, 2, 64, 16, 32)(True, True)[0] is False
    assert parts("bfloat16", 2, 2, 60, 16, 32)(True, True)[0] is False       # rows of weights off 16 bytes
    assert parts("float32", 1, 64, 64, 16, 256)(True, True)[0] is False      # a product that fills the chip
