"""The merge of the latent attention's key splits against float64: split counts around the eight that a wave asks for at once (33 in all) and a wave's
64 lanes, latent dims around the 256 of a workgroup, sizes that 16-byte loads do not take; rows of different split counts in one call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [33, 96, 256, 260, 512])
@pytest.mark.parametrize("splits", [2, 31, 32, 33, 64, 65, 130])
def test_merge_against_float64(r, splits):
    from pegainfer_amd import ops_blocks as B
    H, dr, ps, grain = 2, 32, 16, 32
    g = torch.Generator().manual_seed(r + splits)
    kv = splits * grain - 5
    lens = [kv, 1, kv // 2 + 1]                 # the last key of each is its row's own
    pages = [-(-k // ps) for k in lens]
    pool = torch.randn(sum(pages), ps, r + dr, generator=g)
    qc = torch.randn(len(lens), H, r + dr, generator=g)
    indptr = torch.tensor([sum(pages[:i]) for i in range(len(lens) + 1)], dtype=torch.int32)
    ids = torch.randperm(sum(pages), generator=g).to(torch.int32)
    pos, req = torch.tensor([k - 1 for k in lens], dtype=torch.int32), torch.arange(len(lens), dtype=torch.int32)
    scale = (r + dr) ** -0.5
    got = B.latent_attention(qc.cuda(), pool.cuda(), ps * (r + dr), 0, ps, pos.cuda(), req.cuda(), indptr.cuda(), ids.cuda(), r, dr, scale, kv,
                             split_keys=grain).double().cpu()
    for i, k in enumerate(lens):
        e = pool[ids[indptr[i]:indptr[i + 1]].long()].reshape(-1, r + dr)[:k].double()
        w = (qc[i].double() @ e.t() * scale).softmax(-1)
        # fp32 scores of values of order one over at most 544 products, 2^-24 each, and as many roundings of the weighted sums of up to 4155 keys
        assert float((got[i] - w @ e[:, :r]).abs().max()) < 2e-5
