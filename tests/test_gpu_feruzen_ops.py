"""Every Feruzen mechanism alone on the GPU (torch wrappers of pegainfer_amd/ops_blocks.py over the HIP blocks) against its
function in the plain restatement (oracle/feruzen_ref.py), in both storage types; and crafted inputs where random weights
would hide a fault: one far write among hundreds that a memory has to give back, one far key whose score stands out, keys
on both sides of page and key-tile borders, state regions used by another request before."""
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as Fn

import feruzen_common as C
from oracle import feruzen_ref as R

pytestmark = pytest.mark.gpu

DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
F = torch.float64


def dev(t, dtype):
    return t.to(DT[dtype]).cuda().contiguous()


def close(got, ref, dtype, tol32=2e-5, tol16=3e-2):
    got, ref = got.detach().double().cpu(), ref.double()
    err = float((got - ref).abs().max() / ref.abs().max().clamp_min(1e-9))
    assert err < (tol32 if dtype == "float32" else tol16), err


def B():
    from pegainfer_amd import ops_blocks
    return ops_blocks


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("taps", [1, 2, 5])
def test_time_convolution_carries_its_tail_through_portions_and_slots(dtype, taps):
    g = torch.Generator().manual_seed(taps)
    Cn = 70
    w = C.bf16_round(torch.randn(Cn, taps, generator=g))
    seqs = [C.bf16_round(torch.randn(n, Cn, generator=g)) for n in (23, 9)]
    refs = [x.double() + R.tconv(x.double(), w.double()) for x in seqs]
    state = torch.full((3, max(taps - 1, 1), Cn), 7.0, device="cuda")      # dirty: slots 2 and 0 are zeroed for the new requests
    state[2].zero_()
    state[0].zero_()
    plans = [[(0, 1), (1, 2)], [(0, 2), (1, 1)], [(0, 1), (1, 1)], [(0, 12)], [(0, 7), (1, 5)]]    # (sequence, rows) per step;
    # slots 2 and 0; the third step brings one row per entry: the decode form (output and tail in one launch)
    at, got = [0, 0], [[], []]
    for stp in plans:
        x = torch.cat([seqs[q][at[q]:at[q] + n] for q, n in stp])
        rg = B().Ragged([n for _, n in stp], slots=[2 if q == 0 else 0 for q, _ in stp])
        out = B().time_conv(dev(x, "float32"), dev(w, dtype), state if taps > 1 else state[:, :0], rg, residual=True,
                            out_dtype=torch.float32)
        off = 0
        for q, n in stp:
            got[q].append(out[off:off + n].cpu())
            at[q] += n
            off += n
    for q in range(2):
        close(torch.cat(got[q]), refs[q], "float32", tol32=1e-6)
    assert float(state[1].min()) == 7.0                                      # a slot no entry named is not touched
    x = dev(seqs[0], dtype)                                                  # the mixers' form: stored type in, silu, fp32 out
    state.zero_()
    out = B().time_conv(x, dev(w, dtype), state if taps > 1 else state[:, :0], B().Ragged([23]), silu=True, out_dtype=torch.float32)
    close(out, Fn.silu(R.tconv(seqs[0].double(), w.double())), "float32", tol32=1e-6)


@pytest.mark.parametrize("taps", [1, 3, 4, 7, 8, 9])
def test_time_convolution_over_long_portions(taps):
    """steps of a few hundred rows take the form with a sliding window in registers (up to 8 taps): entries that begin in the
    middle of a thread's walk, a tail carried into the second step, channels beyond a whole workgroup"""
    g = torch.Generator().manual_seed(taps)
    Cn = 300
    w = C.bf16_round(torch.randn(Cn, taps, generator=g))
    seqs = [C.bf16_round(torch.randn(n, Cn, generator=g)) for n in (333, 250, 40)]
    state = torch.zeros(3, max(taps - 1, 1), Cn, device="cuda")
    at, got = [0, 0, 0], [[], [], []]
    for stp in [[(0, 199), (1, 101), (2, 3)], [(2, 37), (0, 134), (1, 149)]]:
        x = torch.cat([seqs[q][at[q]:at[q] + n] for q, n in stp])
        rg = B().Ragged([n for _, n in stp], slots=[q for q, _ in stp])
        out = B().time_conv(dev(x, "bfloat16"), dev(w, "bfloat16"), state if taps > 1 else state[:, :0], rg, silu=True,
                            out_dtype=torch.float32)
        off = 0
        for q, n in stp:
            got[q].append(out[off:off + n].cpu())
            at[q] += n
            off += n
    for q in range(3):
        close(torch.cat(got[q]), Fn.silu(R.tconv(seqs[q].double(), w.double())), "float32", tol32=2e-6)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("mult", [1, 4])        # 4: rows and groups of whole fours take the vector form
@pytest.mark.parametrize("groups", [1, 3, 7])
def test_grouped_output_norm_residual_and_depth_sum(dtype, groups, mult):
    g = torch.Generator().manual_seed(groups)
    d, rows = mult * 42 * groups // math.gcd(42, groups), 9
    y, w = C.bf16_round(torch.randn(rows, d, generator=g) * 3), C.bf16_round(1 + 0.3 * torch.randn(d, generator=g))
    x = torch.randn(rows, d, generator=g)
    stack = torch.randn(3, rows, d, generator=g)
    coef = C.bf16_round(torch.randn(4, generator=g))
    r32, rb, mix = B().group_rms_add(dev(y, dtype), dev(w, dtype), groups, 1e-5, x=x.cuda(), stack=stack.cuda(), coef=dev(coef, dtype))
    ref = x.double() + R.grms(y.double(), w.double(), groups, 1e-5)
    close(r32, ref, "float32", tol32=2e-6)
    close(rb, ref, dtype)
    close(mix, sum(coef[j].double() * stack[j].double() for j in range(3)) + coef[3].double() * ref, "float32", tol32=2e-6)
    only, _, none = B().group_rms_add(dev(y, dtype), dev(w, dtype), groups, 1e-5)     # no residual, no sum: the final norm's form
    close(only, R.grms(y.double(), w.double(), groups, 1e-5), "float32", tol32=2e-6)
    assert none is None


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_clamp_glu(dtype):
    g = torch.Generator().manual_seed(1)
    gu = C.bf16_round(torch.randn(11, 2 * 37, generator=g) * 3)
    out = B().clamp_glu_rows(dev(gu, dtype), 1.25)
    ga, up = gu[:, :37].double().clamp(max=1.25), gu[:, 37:].double().clamp(-1.25, 1.25)
    close(out, ga * torch.sigmoid(1.702 * ga) * (up + 1), dtype)
    assert float(gu[:, :37].min()) < -1.25 and float(out.float().min()) < 0      # the gate is NOT clamped from below


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("experts,top", [(5, 1), (16, 3), (70, 4)])
def test_softmax_router(dtype, experts, top):
    g = torch.Generator().manual_seed(experts)
    h, wr = C.bf16_round(torch.randn(33, 48, generator=g)), C.bf16_round(torch.randn(experts, 48, generator=g) * 0.5)
    e, wt = B().route_topk(dev(h, dtype), dev(wr, dtype), top)
    idx, val = R.router(h.double(), {"r.router": wr}, "r", top)
    assert torch.equal(e.cpu().long().sort(-1).values, idx.sort(-1).values)
    close(wt.cpu().sort(-1).values, val.sort(-1).values, "float32", tol32=1e-5)
    assert float(wt.sum(-1).max()) < 1.0 or top == experts                       # the scores are not renormalised
    # the form the runtime uses: logits by a GEMM into fp32, then the selection alone
    logits = B().linear(dev(h, dtype), dev(wr, dtype), out_dtype=torch.float32)
    e2, w2 = B().route_from_logits(logits, top, dtype=DT[dtype])
    assert torch.equal(e2.cpu().long().sort(-1).values, idx.sort(-1).values)
    close(w2.cpu().sort(-1).values, val.sort(-1).values, "float32", tol32=1e-5)


def run_delta(cfg_m, w, p, h, dtype, lens_plan, eps=1e-5):
    """the delta mixer as the runtime strings it together, rows cut into steps by lens_plan (one request, slot 1)"""
    Bk = B()
    H, G, d, dv, taps = cfg_m["heads"], cfg_m["kv_heads"], cfg_m["dim"], cfg_m["vdim"], cfg_m["conv"]
    Wp = torch.cat([w[p + s] for s in (".q", ".k", ".v", ".g", ".b", ".a")])
    Wc = torch.cat([w[p + s] for s in (".q.conv", ".k.conv", ".v.conv")])
    Cn = 2 * G * d + H * dv
    conv_state = torch.zeros(2, max(taps - 1, 1), Cn, device="cuda")
    mem = torch.full((2, H, d, dv), 3.0, device="cuda")
    mem[1].zero_()
    outs, at = [], 0
    for n in lens_plan:
        rg = Bk.Ragged([n], slots=[1])
        proj = Bk.linear(dev(h[at:at + n], dtype), dev(Wp, dtype), plain=True)
        qkv = Bk.time_conv(proj, dev(Wc, dtype), conv_state if taps > 1 else conv_state[:, :0], rg, silu=True,
                           out_dtype=torch.float32, channels=Cn)
        o = Bk.delta_rule(qkv, proj, Cn + H * dv, Cn + H * dv + H, dev(w[p + ".A_log"], dtype), dev(w[p + ".dt_bias"], dtype), mem,
                          H, G, d, dv, rg)
        mixed = Bk.head_rms_gate(o, dev(w[p + ".norm"], dtype), proj[:, Cn:Cn + H * dv], "silu", 1.0, eps, H, dv)
        outs.append(Bk.linear(mixed, dev(w[p + ".o"], dtype), plain=True))
        at += n
    assert float(mem[0].min()) == 3.0
    return torch.cat(outs)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layer", [("a", 0), ("a", 3), ("wide", 1), ("odd", 1), ("b", 1)])
def test_delta_mixer_whole_and_in_portions(dtype, layer):
    cfg = {"a": C.config_a, "wide": C.config_wide_heads, "odd": C.config_odd, "b": C.config_b}[layer[0]]()
    w = C.random_weights(cfg, 3)
    p, m = "l%d.mix" % layer[1], cfg["layers"][layer[1]]["mixer"]
    h = C.bf16_round(torch.randn(45, cfg["width"], generator=torch.Generator().manual_seed(9)))
    ref = R.delta_mixer(h.double(), w, p, m, 1e-5)
    close(run_delta(m, w, p, h, dtype, [45]), ref, dtype, tol32=1e-4, tol16=6e-2)
    close(run_delta(m, w, p, h, dtype, [1, 2, 17, 1, 16, 8]), ref, dtype, tol32=1e-4, tol16=6e-2)


def test_delta_memory_gives_back_one_far_write_among_hundreds():
    """beta = 1 and no decay: token 3 writes value v* under key e0; 600 later tokens write under the other unit keys, again
    and again; the last token asks with e0 and must read v* (times dim^-1/2), across portions and the staging rounds"""
    Bk = B()
    d, dv, n = 8, 70, 604
    qkv = torch.zeros(n, 2 * d + dv)
    vals = torch.randn(n, dv, generator=torch.Generator().manual_seed(1))
    for t in range(n):
        key = 0 if t == 3 else 1 + (t % (d - 1))
        qkv[t, d + key] = 5.0 if t % 2 else 0.5          # keys of any length: the kernel makes them unit vectors
        qkv[t, key if t < n - 1 else 0] = 2.0
        qkv[t, 2 * d:] = vals[t]
    proj = torch.zeros(n, 2)
    proj[:, 0] = 30.0                                      # beta = sigmoid(30) = 1
    proj[:, 1] = -40.0                                     # softplus(-40) = 0: no decay
    zero = torch.zeros(1, device="cuda")
    for plan in ([n], [2, 1, 300, 1, 299, 1]):
        mem = torch.zeros(1, 1, d, dv, device="cuda")
        outs, at = [], 0
        for k in plan:
            outs.append(Bk.delta_rule(qkv[at:at + k].cuda().contiguous(), proj[at:at + k].cuda().contiguous(), 0, 1, zero, zero,
                                      mem, 1, 1, d, dv, Bk.Ragged([k])))
            at += k
        got = torch.cat(outs)[-1].cpu()
        assert float((got - vals[3] * d ** -0.5).abs().max()) < 1e-4 * float(vals[3].abs().max())


def run_parallel(cfg_m, w, p, h, dtype, plan, page_ids, eps=1e-5, page_size=16):
    """the parallel mixer as the runtime strings it together; plan: rows per step of ONE request whose pages are page_ids"""
    Bk = B()
    a, r = cfg_m["left"], cfg_m["right"]
    H, G, d, dv = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
    H2, d2, dv2 = r["heads"], r["dim"], r["vdim"]
    names = [".left.q", ".left.k", ".left.v", ".right.q", ".right.k", ".right.v", ".right.g", ".right.i", ".right.f"]
    Wp = torch.cat([w[p + s] for s in names])
    offs, at_ = [], 0
    for s in names:
        offs.append(at_)
        at_ += w[p + s].shape[0]
    Wo = torch.cat([w[p + ".left.o"], w[p + ".right.o"]], 1)
    half = a["rot"]["dims"] // 2
    inv_freq = torch.tensor([a["rot"]["base"] ** (-2.0 * i / a["rot"]["dims"]) for i in range(half)] or [0.0], dtype=torch.float32).cuda()
    n_pages = max(page_ids) + 2
    k_off, v_off = 5 * 16, 5 * 16 + page_size * G * d                          # the layer's part does not start the page
    page_stride = v_off + page_size * G * dv + 3
    cache = torch.full((n_pages * page_stride,), float("nan"), dtype=DT[dtype], device="cuda")
    mem = torch.zeros(1, H2 * (d2 * dv2 + d2 + 1), device="cuda")
    indptr = torch.tensor([0, len(page_ids)], dtype=torch.int32, device="cuda")
    pids = torch.tensor(page_ids, dtype=torch.int32, device="cuda")
    outs, at = [], 0
    for n in plan:
        rg = Bk.Ragged([n], starts=[at])
        proj = Bk.linear(dev(h[at:at + n], dtype), dev(Wp, dtype), plain=True)
        q = Bk.qk_norm_rope_paged(proj, offs[:3], H, G, d, dv, dev(w[p + ".left.q.norm"], dtype), dev(w[p + ".left.k.norm"], dtype),
                                  eps, inv_freq, a["rot"]["dims"], rg, indptr, pids, cache, page_stride, k_off, v_off, page_size)
        mix = torch.empty(n, H * dv + H2 * dv2, dtype=DT[dtype], device="cuda")
        mix[:, :H * dv] = Bk.paged_attention(q, cache, page_stride, k_off, v_off, page_size, rg, indptr, pids, G, dv, a["scale"],
                                             cfg_m["left_scale"])
        o = Bk.gated_matrix_memory(proj, offs[3:6] + offs[7:9], dev(w[p + ".right.i.b"], dtype), dev(w[p + ".right.f.b"], dtype),
                                   r["gate_cap"], mem, H2, d2, dv2, rg)
        Bk.head_rms_gate(o, dev(w[p + ".right.norm"], dtype), proj[:, offs[6]:offs[6] + H2 * dv2], "sigmoid", cfg_m["right_scale"],
                         eps, H2, dv2, out=mix[:, H * dv:])
        outs.append(Bk.linear(mix, dev(Wo, dtype), plain=True))
        at += n
    return torch.cat(outs)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layer", [("a", 1), ("a", 2), ("wide", 0), ("wide", 2), ("odd", 0), ("b", 0)])
def test_parallel_mixer_whole_and_in_portions_over_scattered_pages(dtype, layer):
    cfg = {"a": C.config_a, "wide": C.config_wide_heads, "odd": C.config_odd, "b": C.config_b}[layer[0]]()
    w = C.weights_for(cfg, 4, dtype)
    p, m = "l%d.mix" % layer[1], cfg["layers"][layer[1]]["mixer"]
    n = 150
    h = C.bf16_round(torch.randn(n, cfg["width"], generator=torch.Generator().manual_seed(8)))
    ref = R.parallel_mixer(h.double(), w, p, m, 1e-5)
    pages = [7, 2, 11, 0, 5, 9, 3, 12, 1, 10]                                   # ten pages of 16 tokens, in no order
    close(run_parallel(m, w, p, h, dtype, [n], pages), ref, dtype, tol32=1e-4, tol16=6e-2)
    # portions that end just before, at and just after page (16) and key tile (64) borders, then token by token over 127 / 128
    close(run_parallel(m, w, p, h, dtype, [15, 1, 1, 46, 2, 60] + [1] * 25, pages), ref, dtype, tol32=1e-4, tol16=6e-2)


def test_attention_finds_one_far_key_among_hundreds_and_stops_at_the_causal_edge():
    """all keys equal except position 5, whose key points along the last query; its score stands out, so the last row's
    output must be v_5; the row before the marked query has a key of its own kind AFTER it (position 5 + 1 ... are visible,
    the future is not): a second marked key at the very last position must not reach the row before it"""
    Bk = B()
    n, d, dv = 700, 16, 24
    g = torch.Generator().manual_seed(2)
    proj = torch.zeros(n, 2 * d + dv)
    base = torch.randn(d, generator=g)
    mark = torch.randn(d, generator=g)
    mark -= base * (mark @ base) / (base @ base)
    proj[:, :d] = base                               # every query and key looks along `base` ...
    proj[:, d:2 * d] = base
    proj[:, 2 * d:] = torch.randn(n, dv, generator=g)
    proj[5, d:2 * d] = mark * 3                      # ... but key 5 and key n - 1 look along `mark`
    proj[n - 1, d:2 * d] = mark * 3
    proj[n - 2, :d] = mark * 3                       # rows n - 2 and n - 1 ask along `mark`
    proj[n - 1, :d] = mark * 3
    ones = torch.ones(d, device="cuda")
    pages = list(range(44))[::-1]
    indptr = torch.tensor([0, 44], dtype=torch.int32, device="cuda")
    pids = torch.tensor(pages, dtype=torch.int32, device="cuda")
    page_stride = 16 * (d + dv)
    for plan in ([n], [5, 1, 58, 1, 634, 1]):
        cache = torch.zeros(45 * page_stride, device="cuda")
        rows, at = [], 0
        for k in plan:
            rg = Bk.Ragged([k], starts=[at])
            q = Bk.qk_norm_rope_paged(proj[at:at + k].cuda().contiguous(), [0, d, 2 * d], 1, 1, d, dv, ones, ones, 1e-6,
                                      torch.zeros(1, device="cuda"), 0, rg, indptr, pids, cache, page_stride, 0, 16 * d, 16)
            rows.append(Bk.paged_attention(q, cache, page_stride, 0, 16 * d, 16, rg, indptr, pids, 1, dv, 4.0))
            at += k
        out = torch.cat(rows).cpu()
        v = proj[:, 2 * d:]
        assert float((out[n - 2] - v[5]).abs().max()) < 1e-3          # the far key alone; key n - 1 is in this row's future
        assert float((out[n - 1] - 0.5 * (v[5] + v[n - 1])).abs().max()) < 1e-3
        assert float((out[3] - v[:4].mean(0)).abs().max()) < 1e-4     # the first tokens: equal scores, the mean of what is visible


@pytest.mark.parametrize("vdim,steps", [(1040, [1, 1, 2]), (16, [1, 3])])
def test_matrix_memory_workgroups_of_a_head_read_the_same_norm_and_maximum(vdim, steps):
    """a head of 1040 values is dealt over 65 workgroups, and 64 x 8 such heads are more than the chip holds at once: workgroups that begin
    late must not see the vector n and the running maximum that the step leaves"""
    E, H, d = 64, 8, 16
    g = torch.Generator().manual_seed(vdim)
    width = H * (2 * d + vdim + 2)
    offs = [0, H * d, 2 * H * d, 2 * H * d + H * vdim, 2 * H * d + H * vdim + H]
    ib, fb = torch.zeros(H), torch.zeros(H)
    mem = torch.zeros(E, H * (d * vdim + d + 1), device="cuda")
    S, n, m = torch.zeros(E, H, d, vdim, dtype=torch.float64), torch.zeros(E, H, d, dtype=torch.float64), torch.zeros(E, H, dtype=torch.float64)
    for k in steps:
        x = torch.randn(E * k, width, generator=g)
        got = B().gated_matrix_memory(x.cuda(), offs, ib.cuda(), fb.cuda(), 15.0, mem, H, d, vdim, B().Ragged([k] * E))
        xd, ref = x.double().view(E, k, width), []
        for t in range(k):
            q, kk = xd[:, t, :H * d].view(E, H, d) * d ** -0.5, xd[:, t, H * d:2 * H * d].view(E, H, d)
            v = xd[:, t, offs[2]:offs[3]].view(E, H, vdim)
            i = 15 * torch.tanh(xd[:, t, offs[3]:offs[4]] / 15)
            f = Fn.logsigmoid(15 * torch.tanh(xd[:, t, offs[4]:] / 15))
            new = torch.maximum(f + m, i)
            a, b, m = torch.exp(f + m - new), torch.exp(i - new), new
            S = a[..., None, None] * S + b[..., None, None] * kk[..., None] * v[..., None, :]
            n = a[..., None] * n + b[..., None] * kk
            den = torch.maximum((n * q).sum(-1).abs(), torch.exp(-m)) + 1e-6
            ref.append((S * q[..., None]).sum(-2) / den[..., None])
        ref = torch.stack(ref, 1).reshape(E * k, H * vdim)
        close(got, ref, "float32", tol32=2e-5)
        close(mem[:, H * d * vdim:H * d * (vdim + 1)], n.reshape(E, -1), "float32", tol32=2e-6)
        close(mem[:, H * d * (vdim + 1):], m, "float32", tol32=2e-6)


def test_matrix_memory_keeps_a_far_strong_write_and_resets_with_its_slot():
    """token 4 is written with a large input gate, the forget gates stay open: 500 weak writes later its value still
    dominates the read-out; the same slot, zeroed and used by a second request, must not see any of it"""
    Bk = B()
    n, d, dv = 505, 12, 66
    g = torch.Generator().manual_seed(3)
    k = torch.randn(n, d, generator=g)
    v = torch.randn(n, dv, generator=g)
    proj = torch.zeros(n, 2 * d + dv + 2)
    proj[:, :d] = k[4]                               # every query asks for key 4
    proj[:, d:2 * d] = k
    proj[:, 2 * d:2 * d + dv] = v
    proj[:, 2 * d + dv] = -6.0                       # log input gate: weak writes ...
    proj[4, 2 * d + dv] = 9.0                        # ... one strong one
    proj[:, 2 * d + dv + 1] = 20.0                   # forget gate open (logsigmoid(cap tanh(20 / cap)) ~ 0)
    offs = [0, d, 2 * d, 2 * d + dv, 2 * d + dv + 1]
    zero = torch.zeros(1, device="cuda")
    mem = torch.zeros(1, d * dv + d + 1, device="cuda")
    outs, at = [], 0
    for kk in [3, 2, 250, 1, 249]:
        outs.append(Bk.gated_matrix_memory(proj[at:at + kk].cuda().contiguous(), offs, zero, zero, 15.0, mem, 1, d, dv, Bk.Ragged([kk])))
        at += kk
    got = torch.cat(outs)[-1].cpu()
    cos = float(Fn.cosine_similarity(got, v[4], dim=0))
    assert cos > 0.999, cos
    mem.zero_()
    again = Bk.gated_matrix_memory(proj[:3].cuda().contiguous(), offs, zero, zero, 15.0, mem, 1, d, dv, Bk.Ragged([3]))
    assert float((again.cpu() - torch.cat(outs)[:3].cpu()).abs().max()) == 0.0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,dim,vdim", [(2, 128, 256), (3, 16, 8), (1, 20, 33), (2, 256, 130)])
def test_matrix_memory_chunks_against_the_scan_in_64_bits(dtype, heads, dim, vdim):
    """portions around the 64 tokens of a chunk beside one that stays with the scan, a state, its norm and its maximum left from before, odd sizes;
    gates that open and close by turns, so the maximum jumps.  The scan in 64 bits from the stored operands is the reference; outputs are
    quotients, so their error is that of a weighted mean of values of about one."""
    from pegainfer_amd import ops_blocks as Bk
    g = torch.Generator().manual_seed(dim + vdim)
    lens, slots, cap = [64, 3, 65, 320, 127], [1, 4, 0, 3, 5], 15.0
    T, cols = sum(lens), heads * (2 * dim + vdim + 2)
    proj = C.bf16_round(torch.randn(T, cols + 1, generator=g))
    offs = [1, 1 + heads * dim, 1 + 2 * heads * dim, 1 + heads * (2 * dim + vdim), 1 + heads * (2 * dim + vdim + 1)]
    proj[:, offs[3]:] *= 4
    ib, fb = C.bf16_round(torch.randn(heads, generator=g)), C.bf16_round(torch.randn(heads, generator=g) + 2)
    per = heads * (dim * vdim + dim + 1)
    state = torch.randn(6, per, generator=g).cuda()
    before = state.cpu().double()
    td = DT[dtype]
    y = Bk.gated_matrix_memory(proj.cuda().to(td), offs, ib.cuda().to(td), fb.cuda().to(td), cap, state, heads, dim, vdim, Bk.Ragged(lens, slots=slots), scan_max=32)
    y, after, at = y.cpu().double(), state.cpu().double(), 0
    P = proj.double()
    for n, s in zip(lens, slots):
        for h in range(heads):
            S = before[s, h * dim * vdim:(h + 1) * dim * vdim].view(dim, vdim).clone()
            N = before[s, heads * dim * vdim + h * dim:][:dim].clone()
            m = before[s, heads * dim * (vdim + 1) + h].clone()
            for t in range(n):
                row = P[at + t]
                q, k, v = row[offs[0] + h * dim:][:dim] * dim ** -0.5, row[offs[1] + h * dim:][:dim], row[offs[2] + h * vdim:][:vdim]
                i = cap * torch.tanh((row[offs[3] + h] + ib[h].double()) / cap)
                f = torch.nn.functional.logsigmoid(cap * torch.tanh((row[offs[4] + h] + fb[h].double()) / cap))
                mn = torch.maximum(f + m, i)
                a, b = torch.exp(f + m - mn), torch.exp(i - mn)
                S, N, m = a * S + b * torch.outer(k, v), a * N + b * k, mn
                den = torch.maximum((N @ q).abs(), torch.exp(-m)) + 1e-6
                ref = (S.T @ q) / den
                scale = float(((S.abs().T @ q.abs()) / den).max())
                assert float((y[at + t, h * vdim:(h + 1) * vdim] - ref).abs().max()) < 2e-5 * max(1.0, scale), (n, h, t)
            assert float((after[s, h * dim * vdim:(h + 1) * dim * vdim].view(dim, vdim) - S).abs().max()) < 2e-5 * max(1.0, float(S.abs().max()))
            assert float((after[s, heads * dim * vdim + h * dim:][:dim] - N).abs().max()) < 2e-5 * max(1.0, float(N.abs().max()))
            assert abs(float(after[s, heads * dim * (vdim + 1) + h] - m)) < 2e-5 * max(1.0, abs(float(m)))
        at += n
    assert torch.equal(after[2], before[2])


@pytest.mark.parametrize("what", ["value", "key", "query", "gate"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("dim,vdim", [(128, 64), (20, 33)])
def test_matrix_memory_chunks_let_nothing_reach_earlier_tokens(dim, vdim, bad, what):
    """as for the state-space scan: exactly what the token scan spoils is spoilt"""
    from pegainfer_amd import ops_blocks as Bk
    g = torch.Generator().manual_seed(dim)
    heads, T, cap = 2, 150, 15.0
    cols = heads * (2 * dim + vdim + 2)
    offs = [0, heads * dim, 2 * heads * dim, heads * (2 * dim + vdim), heads * (2 * dim + vdim + 1)]
    for at in (16, 45, 63, 64, 121):
        proj = torch.randn(T, cols, generator=g)
        proj[at, {"value": offs[2] + vdim // 2, "key": offs[1] + dim - 1, "query": offs[0] + 2, "gate": offs[4] + 1}[what]] = bad
        ib, fb = torch.randn(heads, generator=g).cuda(), (torch.randn(heads, generator=g) + 2).cuda()
        runs = []
        for scan_max in (0, 32):
            state = torch.zeros(1, heads * (dim * vdim + dim + 1)).cuda()
            y = Bk.gated_matrix_memory(proj.cuda(), offs, ib, fb, cap, state, heads, dim, vdim, Bk.Ragged([T]), scan_max=scan_max)
            runs += [y.cpu(), state.cpu()]
        for a, b in ((runs[0], runs[2]), (runs[1], runs[3])):
            ok = torch.isfinite(a)
            assert torch.equal(ok, torch.isfinite(b)), (at, int((ok != torch.isfinite(b)).sum()))
            assert float((a[ok] - b[ok]).abs().max()) < 1e-4 * max(1.0, float(a[ok].abs().max()))


def test_matrix_memory_chunks_in_runs_of_bounded_scratch():
    """as for the state-space scan, with the keys' own state and the gates of all chunks"""
    from pegainfer_amd import ops_blocks as Bk
    g = torch.Generator().manual_seed(3)
    heads, dim, vdim, lens, slots, cap = 16, 256, 512, [1900, 100, 2300, 20], [2, 0, 3, 1], 15.0
    cols = heads * (2 * dim + vdim + 2)
    offs = [0, heads * dim, 2 * heads * dim, heads * (2 * dim + vdim), heads * (2 * dim + vdim + 1)]
    proj = torch.randn(sum(lens), cols, generator=g).cuda()
    ib, fb = torch.randn(heads, generator=g).cuda(), (torch.randn(heads, generator=g) + 2).cuda()
    runs = []
    for scan_max in (0, 64):
        state = torch.zeros(4, heads * (dim * vdim + dim + 1)).cuda()
        runs.append((Bk.gated_matrix_memory(proj, offs, ib, fb, cap, state, heads, dim, vdim, Bk.Ragged(lens, slots=slots), scan_max=scan_max), state))
    # outputs are quotients by a sum that can be small: those of a typical size agree to rounding, all of them to a few units of it
    (a, sa), (b, sb) = runs
    assert float((sa - sb).abs().max()) < 2e-5 * float(sa.abs().max())
    err = (a - b).abs() / (1 + a.abs())
    assert float(err.mean()) < 1e-5 and float(err.max()) < 2e-2


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("d,groups", [(4, 1), (1024, 4), (1028, 1), (2560, 5), (4096, 64), (4100, 5), (8192, 2)])
def test_row_step_joins_norms_mixes_and_convolves(dtype, d, groups):
    """both norms, a stored output or the routed sum with its added rows (stored or in parts), streams mixed, four taps with their tails moved on in
    scattered slots: against double precision; fp32 sums of d values, a bf16 result rounded once"""
    import importlib
    B = importlib.import_module("pegainfer_amd.ops_blocks")
    g = torch.Generator().manual_seed(d + groups)
    rows, top, n_add, n_mix, eps, dt = 3, 2, 2, 4, 1e-5, getattr(torch, dtype)
    f32 = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    st = lambda *s: torch.randn(*s, generator=g).to(dt)  # noqa: E731
    x, y, bias, vec, extra, gain, one = f32(rows, d), st(rows, d), st(d), st(d), f32(rows, d), st(d), st(1)
    pairs, wt, gate, add, parts = f32(rows * top, d), torch.rand(rows, top, generator=g), f32(rows, 3), st(rows, d), f32(n_add, rows, d)
    stack, coef, cw = f32(n_mix - 1, rows, d), st(n_mix), st(d, 4)
    slots, stride = torch.tensor([2, 0, 3], dtype=torch.int32), 3 * d + 8
    state = f32(4, stride)
    routed = (wt.double()[:, :, None] * pairs.double().view(rows, top, d)).sum(1)
    sig = torch.sigmoid(gate[:, 1:2].double())

    def close_(got, ref, stored):
        tol = 4e-6 * ref.abs().max() + (ref.abs() * 2.0 ** -8 if stored and dtype == "bfloat16" else 0)
        assert bool(((got.cpu().double() - ref).abs() <= tol).all())

    def conv(n, out, sd):
        tail = state[slots.long(), 4:4 + 3 * d].view(rows, 3, d).double()
        close_(out, n + (torch.cat([tail, n[:, None]], 1) * cw.double().T[None]).sum(1), True)
        want = state.clone().double()
        want[slots.long(), 4:4 + 3 * d] = torch.cat([tail[:, 1:], n[:, None]], 1).reshape(rows, -1)
        close_(sd, want, False)
    for kind in ("stored", "routed", "parts"):
        src = dict(y=y.cuda(), bias=bias.cuda()) if kind == "stored" else dict(y_pairs=pairs.cuda(), weight=wt.cuda(), top=top)
        v = y.double() + bias.double() if kind == "stored" else routed
        if kind != "stored":
            gd = gate.cuda()
            src.update(add_gate=gd[:, 1], add_gate_stride=3)
            src.update(dict(add=add.cuda()) if kind == "routed" else dict(add_pairs=parts.cuda(), n_add=n_add))
            v = v + sig * (add.double() if kind == "routed" else parts.double().sum(0))
        for grouped in (False, True):
            sd, xo, out = state.cuda(), x.cuda(), torch.zeros(rows, d, dtype=dt, device="cuda")
            cv = dict(conv_w=cw.cuda(), conv_state=sd[0, 4:], conv_slot_stride=stride, conv_slot=slots.cuda(), conv_out=out)
            if grouped:
                xb, mix = torch.zeros(rows, d, dtype=dt, device="cuda"), torch.zeros(rows, d, device="cuda")
                sk, cf, gn = stack.cuda(), coef.cuda(), gain.cuda()
                B.row_step(dt, rows, d, x_in=xo, x_out=xo, gain=gn, groups=groups, eps=eps, xb_out=xb, stack=sk, stack_stride=rows * d, coef=cf, n_mix=n_mix,
                           mix_out=mix, **src, **cv)
                vn = v.view(rows, groups, -1)
                r = x.double() + (vn / torch.sqrt((vn * vn).mean(-1, keepdim=True) + eps)).view(rows, d) * gain.double()
                n = (coef.double()[:-1, None, None] * stack.double()).sum(0) + coef.double()[-1] * r
                close_(xb, r, True)
                close_(mix, n, False)
            else:
                no, ex, vc, on = torch.zeros(rows, d, device="cuda"), extra.cuda(), vec.cuda(), one.cuda()
                B.row_step(dt, rows, d, x_in=xo, x_out=xo, mult=0.3, add_rows=ex, add_vec=vc, gain=on, eps=eps, n_out=no, **src, **cv)
                r = x.double() + 0.3 * v + extra.double() + vec.double()
                n = r / torch.sqrt((r * r).mean(-1, keepdim=True) + eps) * one.double()
                close_(no, n, False)
            close_(xo, r, False)
            conv(n, out, sd)
    pick, no, xd, on = torch.tensor([2, 2, 0, 1, 2], dtype=torch.int32).cuda(), torch.zeros(5, d, device="cuda"), x.cuda(), one.cuda()
    B.row_step(dt, 5, d, x_in=xd, row_index=pick, gain=on, eps=eps, n_out=no)
    close_(no, (x.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + eps) * one.double())[pick.cpu().long()], False)


def test_row_step_refuses_what_its_form_leaves_out():
    """parts of the other form, a bias without an output to add it to, and rows picked from the matrix that is written: an error, and nothing is written"""
    import importlib
    B = importlib.import_module("pegainfer_amd.ops_blocks")
    rows, d, dt = 3, 64, torch.bfloat16
    ones = lambda *s, t=torch.float32: torch.ones(*s, dtype=t, device="cuda")  # noqa: E731
    x, other, y, vec, pairs, weight = ones(rows, d), ones(rows, d), ones(rows, d, t=dt), ones(d, t=dt), ones(rows, d), ones(rows, 1)
    pick = torch.tensor([2, 0, 1], dtype=torch.int32, device="cuda")
    grouped, scalar = dict(x_in=x, x_out=x, y=y, gain=vec, groups=4, eps=1e-5), dict(x_in=x, x_out=x, y=y, gain=vec, eps=1e-5)
    routed = dict(x_in=x, x_out=x, y_pairs=pairs, weight=weight, top=1, gain=vec, eps=1e-5)
    for form, part in ([(grouped, p) for p in (dict(row_index=pick), dict(add_rows=other), dict(add_vec=vec), dict(n_out=other))] +
                       [(scalar, p) for p in (dict(stack=other), dict(coef=vec), dict(mix_out=other), dict(xb_out=y), dict(row_index=pick))] +
                       [(routed, dict(bias=vec)), (dict(routed, groups=4), dict(bias=vec)), (dict(scalar, y=None), dict(bias=vec))]):
        with pytest.raises(RuntimeError):
            B.row_step(dt, rows, d, **{k: v for k, v in dict(form, **part).items() if v is not None})
        torch.cuda.synchronize()
        assert all(bool((t == 1).all()) for t in (x, other, y, vec))
    for form in (scalar, grouped, routed):
        B.row_step(dt, rows, d, **dict(form, x_out=other))
    B.row_step(dt, rows, d, **dict(scalar, row_index=pick, x_out=other))
