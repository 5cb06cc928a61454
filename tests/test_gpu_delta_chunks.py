"""The delta rule 16 tokens at a time against float64, token by token: entries around whole chunks (and empty ones), every number of rows of S a wave
holds, more value heads per key head than are prepared side by side, decays from none to all at once, a state carried on by the token-by-token form."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def reference(qkv, g, beta, S, H, G, d, dv):
    q, k, v = qkv[:, :G * d].view(-1, G, d), qkv[:, G * d:2 * G * d].view(-1, G, d), qkv[:, 2 * G * d:].view(-1, H, dv)
    q, k = ((t / (t.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()).repeat_interleave(H // G, 1) for t in (q, k))
    out = []
    for t in range(len(q)):
        S = S * g[t].view(H, 1, 1)
        u = beta[t].view(H, 1) * (v[t] - (S * k[t][..., None]).sum(1))
        S = S + k[t][..., None] * u[:, None]
        out.append((S * q[t][..., None]).sum(1).reshape(-1) * d ** -0.5)
    return (torch.stack(out) if out else qkv.new_zeros(0, H * dv)), S


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("gate", [-40.0, -3.0, 3.0, 200.0])        # no decay, slow, fast, all at once
@pytest.mark.parametrize("H,G,d,dv,lens", [(2, 1, 64, 16, [1, 0, 16]), (6, 6, 128, 48, [17, 15, 2]), (12, 2, 128, 16, [0, 33, 48]), (5, 1, 192, 32, [49, 31]),
                                           (4, 4, 256, 16, [64, 5, 80, 1])])
def test_chunks_against_float64(dtype, gate, H, G, d, dv, lens):
    from pegainfer_amd import ops_blocks as B
    gen = torch.Generator().manual_seed(H * d + len(lens))
    n, T, dt = len(lens), sum(lens), DT[dtype]
    slots = torch.randperm(n + 1, generator=gen)[:n]
    mem = torch.randn(n + 1, H, d, dv, generator=gen)
    A_log, bias = (torch.randn(H, generator=gen) * 0.3).to(dt), (torch.randn(H, generator=gen) * 0.3).to(dt)
    S, st = mem.double(), mem.cuda()
    for step in range(2):                                          # the second one through the token-by-token form
        qkv = torch.randn(T, 2 * G * d + H * dv, generator=gen)
        qkv[1:, G * d:2 * G * d] = 0.6 * qkv[:-1, G * d:2 * G * d] + 0.8 * qkv[1:, G * d:2 * G * d]
        proj = torch.randn(T, 2 * H + 3, generator=gen).to(dt)
        proj[:, H:2 * H] += gate
        p64 = proj.double()
        g = torch.exp(-A_log.double().exp() * torch.nn.functional.softplus(p64[:, H:2 * H] + bias.double()))
        rg = B.Ragged(lens, slots=slots.tolist())
        got = B.delta_rule(qkv.cuda(), proj.cuda(), 0, H, A_log.cuda(), bias.cuda(), st, H, G, d, dv, rg, chunked=step == 0)
        at = 0
        for e, (length, slot) in enumerate(zip(lens, slots.tolist())):
            rows = slice(at, at + length)
            ref, S[slot] = reference(qkv[rows].double(), g[rows], torch.sigmoid(p64[rows, :H]), S[slot], H, G, d, dv)
            at += length
            if length:      # sums of up to 256 fp32 products, 2^-24 each, through a triangle of up to 16 and some chunks: 1e-5 of the largest value
                assert float((got[rows].double().cpu() - ref).abs().max() / ref.abs().max()) < 1e-5, (step, e)
            assert float((st[slot].double().cpu() - S[slot]).abs().max() / S[slot].abs().max()) < 1e-5, (step, e)
    untouched = [i for i in range(n + 1) if i not in slots.tolist()]
    assert torch.equal(st[untouched].cpu(), mem[untouched])


def test_sizes_that_are_left_to_the_token_form():
    from pegainfer_amd import ops_blocks as B
    for d, dv in ((32, 16), (128, 24), (320, 16)):
        qkv, z = torch.zeros(20, 2 * d + dv, device="cuda"), torch.zeros(1, device="cuda")
        assert B.delta_rule(qkv, torch.zeros(20, 2, device="cuda"), 0, 1, z, z, torch.zeros(1, 1, d, dv, device="cuda"), 1, 1, d, dv, B.Ragged([20]),
                            chunked=True) is None


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("what", ["value", "key", "query", "beta", "decay"])
@pytest.mark.parametrize("H,G,d,dv", [(2, 1, 64, 32), (3, 3, 192, 16)])
def test_chunks_let_nothing_reach_earlier_tokens(H, G, d, dv, what, bad):
    """exactly what the token-by-token form spoils is spoilt: from the token on, in its column or head, the state included; the rest stays within
    the two forms' rounding of each other (1e-5 each of the largest value)"""
    from pegainfer_amd import ops_blocks as B
    gen = torch.Generator().manual_seed(d)
    T = 47                                                         # two whole chunks and one that repeats its last row
    A, bias, mem = torch.zeros(H), torch.zeros(H), torch.randn(1, H, d, dv, generator=gen)
    for at in (0, 9, 15, 16, 38, 46):
        qkv, proj = torch.randn(T, 2 * G * d + H * dv, generator=gen), torch.randn(T, 2 * H, generator=gen)
        if what in ("beta", "decay"):
            proj[at, H - 1 if what == "beta" else 2 * H - 1] = bad
        else:
            qkv[at, {"query": 3, "key": 2 * G * d - 1, "value": 2 * G * d + dv + 5}[what]] = bad
        runs = []
        for chunked in (False, True):
            st = mem.cuda()
            runs.append((B.delta_rule(qkv.cuda(), proj.cuda(), 0, H, A.cuda(), bias.cuda(), st, H, G, d, dv, B.Ragged([T]), chunked=chunked).cpu(), st.cpu()))
        for a, b in zip(*runs):
            ok = torch.isfinite(a)
            assert torch.equal(ok, torch.isfinite(b)), (at, int((ok != torch.isfinite(b)).sum()))
            if ok.any():
                assert float((a[ok] - b[ok]).abs().max()) < 2e-5 * float(a[ok].abs().max()), at


@pytest.mark.parametrize("G,d,dv", [(2, 128, 32), (3, 64, 16), (6, 256, 16), (1, 192, 48)])
@pytest.mark.parametrize("lens,scan_max", [([1, 30, 200, 64, 0, 65], 64), ([17, 3, 16], 16), ([5, 6], 64), ([70, 90], 64)])
def test_an_entry_takes_the_form_of_its_own_length(G, d, dv, lens, scan_max):
    """outputs, states and the rows made unit vectors: the bits that each entry has alone, token by token up to scan_max tokens and in chunks beyond"""
    from pegainfer_amd import ops_blocks as B
    H = 6
    gen = torch.Generator().manual_seed(len(lens))
    n, T = len(lens), sum(lens)
    A, bias = torch.randn(H, generator=gen).cuda(), torch.randn(H, generator=gen).cuda()
    qkv0, proj, mem = torch.randn(T, 2 * G * d + H * dv, generator=gen).cuda(), torch.randn(T, 2 * H, generator=gen).cuda(), torch.randn(n, H, d, dv, generator=gen).cuda()
    qkv, st = qkv0.clone(), mem.clone()
    got = B.delta_rule(qkv, proj, 0, H, A, bias, st, H, G, d, dv, B.Ragged(lens), chunked=True, scan_max=scan_max)
    at = 0
    for e, length in enumerate(lens):
        rows, at = slice(at, at + length), at + length
        if length == 0:
            assert torch.equal(st[e], mem[e])
            continue
        own, own_st = qkv0[rows].clone(), mem[e:e + 1].clone()
        alone = B.delta_rule(own, proj[rows].clone(), 0, H, A, bias, own_st, H, G, d, dv, B.Ragged([length]), chunked=length > scan_max)
        assert torch.equal(got[rows], alone) and torch.equal(st[e], own_st[0]) and torch.equal(qkv[rows], own), e


def test_a_long_step_in_runs_of_bounded_scratch():
    """256 MB hold 455 chunks of 256 heads: the last entry's lie on both sides of the cut, and have the bits of a run of their own"""
    from pegainfer_amd import ffi
    from pegainfer_amd import ops_blocks as B
    need = ffi.lib().pegainfer_delta_rule_workspace
    assert need(10 ** 6, 1, 32) * 4 <= 256 << 20 and need(10 ** 6, 9, 32) == need(2 * 10 ** 6, 9, 32) and need(1, 1, 10 ** 6) >= 10 ** 6
    H, G, d, dv, lens = 256, 1, 64, 16, [7000, 40, 900]
    assert need(sum(lens), len(lens), H) < need(sum(lens), len(lens), H // 2) * 2
    g = torch.Generator(device="cuda").manual_seed(1)
    T = sum(lens)
    qkv, proj = (torch.randn(T, w, device="cuda", generator=g) for w in (2 * G * d + H * dv, 2 * H))
    A, bias, mem = torch.zeros(H, device="cuda"), torch.full((H,), -3.0, device="cuda"), torch.randn(3, H, d, dv, device="cuda", generator=g)
    st, own_st = mem.clone(), mem[2:].clone()
    own, own_proj = qkv[-900:].clone(), proj[-900:].clone()
    got = B.delta_rule(qkv, proj, 0, H, A, bias, st, H, G, d, dv, B.Ragged(lens), chunked=True)
    alone = B.delta_rule(own, own_proj, 0, H, A, bias, own_st, H, G, d, dv, B.Ragged([900]), chunked=True)
    assert torch.equal(got[-900:], alone) and torch.equal(st[2], own_st[0])
