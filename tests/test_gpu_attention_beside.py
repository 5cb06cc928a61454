"""A decode step of a recurrence in the launch of a paged attention: the same bits as the two launches one after the other, for every width of
values, whole and split keys, a recurrence with more and with fewer workgroups than the attention; and the forms that take none."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def parts(n, H, G, d, heads, dim, vdim, seed=0):
    """(attend(beside, **kw), step(launch) -> (its description or None, read-out), the recurrence's state)"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(seed + n * d + dim)
    draw = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    starts = [int(t) for t in torch.randint(0, 300, (n,), generator=g)]
    pages = [-(-(t + 1) // 16) for t in starts]
    stride = 2 * 16 * G * d
    cache = draw(sum(pages), stride)
    indptr = torch.tensor([sum(pages[:i]) for i in range(n + 1)], dtype=torch.int32).cuda()
    pids = torch.randperm(sum(pages), generator=g).to(torch.int32).cuda()
    rg = B.Ragged([1] * n, starts=starts)
    q = torch.randn(n, H, d, generator=g).cuda()
    state, slots = torch.randn(n, heads * dim * vdim, generator=g).cuda(), torch.randperm(n, generator=g).to(torch.int32).cuda()
    width = -(-(heads * (2 * dim + 2 * vdim)) // 8) * 8
    proj, norm_w, z, bias = draw(n, width), draw(vdim), torch.randn(n, heads * dim, generator=g).cuda(), draw(heads * dim)
    offs = [heads * vdim, heads * (vdim + dim), 0]

    def step(launch=True):
        return B.recurrent_step("gated", proj, offs, proj, state, slots, norm_w, heads, heads, dim, vdim, q_scale=dim ** -0.5, z=z, z_bias=bias, tau=4.0,
                                gate=proj[:, heads * (vdim + 2 * dim):], launch=launch)

    def attend(beside=None, **kw):
        return B.paged_attention_opt(q, cache, stride, 0, 16 * G * d, 16, rg, indptr, pids, G, d, d ** -0.5, beside=beside, **kw)

    return attend, step, state


@pytest.mark.parametrize("n_split", [1, 7])
@pytest.mark.parametrize("n,H,G,d,heads,dim,vdim", [(1, 2, 1, 32, 1, 16, 4), (3, 6, 2, 64, 5, 100, 68), (2, 4, 4, 128, 2, 128, 128), (5, 3, 1, 256, 1, 33, 124),
                                                    (9, 8, 8, 128, 1, 64, 64)])
def test_both_as_by_themselves(n_split, n, H, G, d, heads, dim, vdim):
    attend, step, state = parts(n, H, G, d, heads, dim, vdim)
    before = state.clone()
    a, s, after = attend(n_split=n_split), step(), state.clone()
    state.copy_(before)
    desc, out = step(launch=False)
    got = attend(beside=desc, n_split=n_split)
    assert torch.equal(got, a) and torch.equal(out, s) and torch.equal(state, after)
    assert torch.isfinite(s.float()).all() and s.float().abs().max() > 0


def test_forms_that_take_no_step():
    attend, step, state = parts(2, 2, 1, 64, 2, 64, 64)
    before = state.clone()
    desc, _ = step(launch=False)
    assert attend(beside=desc, plain=True) is None
    for field, value in (("kind", 1), ("dtype", 0 if desc.dtype else 1), ("vdim", 66), ("n_entries", 0)):
        old = getattr(desc, field)
        setattr(desc, field, value)
        assert attend(beside=desc) is None, field
        setattr(desc, field, old)
    assert torch.equal(state, before)
