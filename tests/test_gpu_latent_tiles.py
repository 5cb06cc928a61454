"""The prompts' form of the latent attention (whole blocks of 32 values, pages of a multiple of eight keys) against float64: key counts around its tiles of
64, row counts around its blocks of 16, contexts before the portion, keys split between workgroups, tiles in any order, all keys alike but one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def attend(lens, starts, H, r, dr, ps, split_keys=4096, hot=None, seed=0, swap=False):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(seed + r + dr + sum(lens))
    E, T, n = r + dr, sum(lens), len(lens)
    ents = [torch.randn(s + k, E, generator=g).bfloat16() for s, k in zip(starts, lens)]
    qc = torch.randn(T, H, E, generator=g)
    if hot is not None:
        ents = [torch.full_like(e, 0.01) for e in ents]
        for e in ents:
            e[hot, :r] = 1.0
        qc = qc.abs()
    pages = [-(-len(e) // ps) for e in ents]
    ids = torch.randperm(sum(pages) + 2, generator=g)[:sum(pages)].to(torch.int32)
    pool = torch.full((sum(pages) + 2, ps, E), float("nan"), dtype=torch.bfloat16)
    at = 0
    for e, p in zip(ents, pages):
        for k in range(len(e)):
            pool[ids[at + k // ps], k % ps] = e[k]
        at += p
    indptr = torch.tensor([sum(pages[:i]) for i in range(n + 1)], dtype=torch.int32)
    pos = torch.cat([torch.arange(s, s + k) for s, k in zip(starts, lens)]).int()
    req = torch.cat([torch.full((k,), i) for i, k in enumerate(lens)]).int()
    row0, rows = B.row_tiles(lens, H)
    if swap:
        row0, rows = row0.flip(0).contiguous(), rows.flip(0).contiguous()
    scale = E ** -0.5
    got = B.latent_attention(qc.cuda(), pool.cuda(), ps * E, 0, ps, pos.cuda(), req.cuda(), indptr.cuda(), ids.cuda(), r, dr, scale,
                             max(len(e) for e in ents), split_keys=split_keys, tiles=(row0, rows)).double().cpu()
    ref, at = [], 0
    for e, s, k in zip(ents, starts, lens):
        q = qc[at:at + k].bfloat16().double()
        sc = torch.einsum("thd,jd->thj", q, e.double()) * scale
        sc = sc.masked_fill((torch.arange(s + k)[None] > torch.arange(s, s + k)[:, None])[:, None], float("-inf"))
        ref.append(torch.einsum("thj,jd->thd", sc.softmax(-1), e[:, :r].double()))
        at += k
    return got, torch.cat(ref)


@pytest.mark.parametrize("r,dr", [(256, 32), (256, 64), (512, 32), (512, 64)])
@pytest.mark.parametrize("lens,starts,H,ps", [([64], [0], 2, 16), ([17, 3], [0, 63], 3, 8), ([40, 1, 5], [1, 0, 200], 16, 24), ([9], [119], 7, 16)])
def test_prompts_against_float64(r, dr, lens, starts, H, ps):
    # weights and the row sum in bf16 (2^-9 each, one against the other), of values of order one: 4 / 512 of the largest at most
    for split_keys, swap in ((4096, False), (64, True)):
        got, ref = attend(lens, starts, H, r, dr, ps, split_keys, swap=swap)
        assert float((got - ref).abs().max() / ref.abs().max()) < 8e-3


@pytest.mark.parametrize("hot", [0, 63, 64, 130])
def test_one_key_that_stands_out(hot):
    got, ref = attend([40], [120], 4, 512, 64, 16, hot=hot)
    assert float((got - ref).abs().max() / ref.abs().max()) < 8e-3
    assert float(ref[20].max()) > 0.5
