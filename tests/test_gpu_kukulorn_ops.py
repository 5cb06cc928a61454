"""Every Kukulorn mechanism alone on the GPU (torch wrappers of pegainfer_amd/ops_blocks.py over the HIP blocks) against its
function in the plain restatement (oracle/kukulorn_ref.py), in both storage types; and crafted inputs where random weights would
hide a fault: one far key whose score stands out among hundreds, marked keys just inside and just outside the window and the kept
first tokens in prompts and in decoding, a soft cap that binds, a distance bias that decides the softmax, a state that one old
token wrote and a fast decay forgets, state regions and pages used by another request before."""
import math

import numpy as np
import pytest
import torch

import kukulorn_common as C
from oracle import kukulorn_ref as R

pytestmark = pytest.mark.gpu

DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
F = torch.float64


def dev(t, dtype):
    return t.to(DT[dtype]).cuda().contiguous()


def close(got, ref, dtype, tol32=2e-5, tol16=3e-2):
    got, ref = got.detach().double().cpu(), ref.double()
    err = float((got - ref).abs().max() / ref.abs().max().clamp_min(1e-9))
    assert err < (tol32 if dtype == "float32" else tol16), err


def close_rows(got, ref, dtype, tol32=1e-4, tol16=6e-2):
    """fp32: every value.  bf16: per row; one row in fifty (or one) may be off by more.  A single-headed state-space layer reads
    y = (dt B.C + D) x through a norm that forgets its scale: where that factor happens to cancel, rounding the projection to bf16
    moves the restatement itself by 8 % (measured on the CPU); a fault that hits single rows is the fp32 run's to find."""
    if dtype == "float32":
        return close(got, ref, dtype, tol32=tol32)
    got, ref = got.detach().double().cpu(), ref.double()
    err = (got - ref).abs().max(-1).values / ref.abs().max().clamp_min(1e-9)
    assert float(err.median()) < tol16 / 2 and int((err > tol16).sum()) <= max(1, err.numel() // 50), (float(err.median()), float(err.max()))


def B():
    from pegainfer_amd import ops_blocks
    return ops_blocks


def w64(w):
    return {k: v.double() for k, v in w.items()}


# ------------------------------------------------------------------ norms, sums, activations
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("d", [50, 1024, 1300, 5000, 9001])        # one to thirty-two values per thread, then the two-pass form
def test_sum_of_normed_and_plain_terms_then_norm(dtype, d):
    g = torch.Generator().manual_seed(d)
    rows, eps = 5, 1e-6
    x = torch.randn(rows, d, generator=g) * 3
    y1, y2, y3, b1, w1, w2, gain = (C.bf16_round(torch.randn(*s, generator=g)) for s in
                                    ((rows, d), (rows, d), (rows, d), (d,), (d,), (d,), (d,)))
    terms = [(dev(y1, dtype), dev(b1, dtype), dev(w1, dtype), 0.5), (dev(y2, dtype), None, dev(w2, dtype), 0.5), (dev(y3, dtype), None, None, 1.0)]
    r, n = B().terms_rms_add(x.cuda(), terms, gain=dev(gain, dtype), eps=eps, out_dtype=torch.float32)
    ref = x.double() + 0.5 * R.rms(y1.double() + b1.double(), eps) * w1.double() + 0.5 * R.rms(y2.double(), eps) * w2.double() + y3.double()
    close(r, ref, "float32", tol32=3e-6)
    close(n, R.rms(ref, eps) * gain.double(), "float32", tol32=3e-6)
    r, n = B().terms_rms_add(x.cuda(), [], gain=dev(gain, dtype), eps=eps)                   # the norm alone, stored type out
    close(n, R.rms(x.double(), eps) * gain.double(), dtype, tol32=3e-6, tol16=1e-2)
    r, n = B().terms_rms_add(x.cuda(), terms[2:], gain=None)                                 # the sum alone
    close(r, x.double() + y3.double(), "float32", tol32=3e-6)
    assert n is None
    wide = dev(torch.cat([y1, y3], 1), dtype)                                                # a term that is a column range
    r, _ = B().terms_rms_add(x.cuda(), [(wide[:, d:], None, None, 2.0)], gain=None)
    close(r, x.double() + 2.0 * y3.double(), "float32", tol32=3e-6)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,d", [(1, 64), (3, 260), (255, 2048), (256, 2048), (2, 4096), (2, 4100), (3, 1026)])
def test_terms_of_few_and_many_rows(dtype, rows, d):
    # below 256 rows of up to 4096 columns in fours a row is one pass of its workgroup; the other shapes take the general form
    g = torch.Generator().manual_seed(rows + d)
    x = torch.randn(rows, d, generator=g)
    y1, y2, y3 = (C.bf16_round(torch.randn(rows, d, generator=g)) for _ in range(3))
    w1, w3, b1, gain = (C.bf16_round(torch.randn(d, generator=g)) for _ in range(4))
    terms = [(dev(y1, dtype), dev(b1, dtype), dev(w1, dtype), 0.5), (dev(y2, dtype), None, None, -2.0), (dev(y3, dtype), None, dev(w3, dtype), 1.0)]
    r, n = B().terms_rms_add(x.cuda(), terms, gain=dev(gain, dtype), eps=1e-5, out_dtype=torch.float32)
    ref = x.double() + 0.5 * R.rms(y1.double() + b1.double(), 1e-5) * w1.double() - 2 * y2.double() + R.rms(y3.double(), 1e-5) * w3.double()
    close(r, ref, "float32", tol32=3e-6)
    close(n, R.rms(ref, 1e-5) * gain.double(), "float32", tol32=3e-6)
    pick = torch.randint(0, rows, (rows,), generator=g, dtype=torch.int32)
    dt = DT[dtype]
    r, n = B().terms_rms(dt, d, x=x.cuda(), row_index=pick.cuda(), gain=dev(gain, dtype), eps=1e-5, gain_offset=1.0)
    close(n, R.rms(x[pick.long()].double(), 1e-5) * (1 + gain.double()), dtype, tol32=3e-6, tol16=4e-3)
    emb, pairs = C.bf16_round(torch.randn(11, d, generator=g)), C.bf16_round(torch.randn(8, d, generator=g))
    ids = torch.randint(0, 11, (rows,), generator=g)
    prev = torch.randint(-1, 11, (rows,), generator=g)
    r, n = B().terms_rms(dt, d, embed=dev(emb, dtype), token_ids=ids.to(torch.int32).cuda().view(torch.uint32), embed_scale=1.5,
                         pair_table=dev(pairs, dtype), prev_ids=prev.to(torch.int32).cuda(), muls=(5, 3), gain=dev(gain, dtype), eps=1e-5)
    at = torch.where(prev < 0, torch.full_like(prev, 7), (prev * 5 + ids * 3) % 7)
    ref = emb[ids].double() * 1.5 + pairs[at].double()
    close(r, ref, "float32", tol32=1e-6)
    close(n, R.rms(ref, 1e-5) * gain.double(), dtype, tol32=3e-6, tol16=4e-3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("channels,taps,I", [(300, 4, 257), (256, 1, 40), (70, 8, 300), (33, 10, 7)])
def test_convolution_step_with_a_gated_unit_beside_it(dtype, channels, taps, I):
    g = torch.Generator().manual_seed(channels)
    n = 5
    rows = C.bf16_round(torch.randn(n, channels + 2 * I + 3, generator=g))
    w, ib, ob = (C.bf16_round(torch.randn(*s, generator=g)) for s in ((channels, taps), (channels,), (channels,)))
    state = torch.randn(6, max(taps - 1, 1), channels, generator=g)
    d, st, rg = dev(rows, dtype), state.cuda(), B().Ragged([1] * n, slots=[4, 0, 5, 2, 1])
    conv, glu = B().conv_glu_step(d[:, :channels], dev(w, dtype), st, rg, d[:, channels:channels + I], d[:, channels + I:channels + 2 * I], "silu",
                                  silu=True, in_bias=dev(ib, dtype), out_bias=dev(ob, dtype))
    close(glu, R.silu(rows[:, channels:channels + I].double()) * rows[:, channels + I:channels + 2 * I].double(), dtype, tol32=2e-6, tol16=4e-3)
    for e, slot in enumerate((4, 0, 5, 2, 1)):
        past = torch.cat([state[slot, :taps - 1].double(), (rows[e:e + 1, :channels] + ib).double()])
        close(conv[e], R.silu((past * w.double().t()).sum(0) + ob.double()), "float32", tol32=2e-6)
        if taps > 1:
            close(st[slot], past[1:], "float32", tol32=1e-6)
    assert torch.equal(st[3].cpu(), state[3])


def test_embedding_rows_beside_themselves():
    emb = torch.randn(9, 300).bfloat16().cuda()
    ids = torch.tensor([3, 8, 3, 0], dtype=torch.int32).cuda().view(torch.uint32)
    out, pair = B().embed_f32_pair(emb, ids)
    ref = emb[torch.tensor([3, 8, 3, 0]).cuda()].float()
    assert torch.equal(out, ref) and torch.equal(pair, torch.cat([ref, ref], 1))
    none, pair = B().embed_f32_pair(emb, ids, stream=False)
    assert none is None and torch.equal(pair, torch.cat([ref, ref], 1))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_glu_activations_and_soft_cap(dtype):
    g = torch.Generator().manual_seed(1)
    gu = C.bf16_round(torch.randn(7, 2 * 37 + 5, generator=g) * 2)
    d = dev(gu, dtype)
    gate, up = gu[:, :37].double(), gu[:, 40:77].double()
    for act, fn in (("relu", torch.relu), ("silu", lambda t: t * torch.sigmoid(t)),
                    ("gelu_tanh", lambda t: 0.5 * t * (1 + torch.tanh(math.sqrt(2 / math.pi) * (t + 0.044715 * t ** 3))))):
        close(B().glu_rows(d[:, :37], d[:, 40:77], act), fn(gate) * up, dtype, tol16=1e-2)
    x = torch.randn(3, 1000, generator=g) * 40
    close(B().softcap_rows(x.cuda(), 30.0), 30.0 * torch.tanh(x.double() / 30.0), "float32", tol32=1e-6)
    assert float(B().softcap_rows(x.cuda(), 30.0).abs().max()) <= 30.0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", [(3, 16), (1, 100), (5, 7), (2, 200)])
def test_gate_before_the_norm_in_groups(dtype, shape):
    heads, vd = shape
    g = torch.Generator().manual_seed(heads)
    o = torch.randn(9, heads * vd, generator=g)
    z, w = C.bf16_round(torch.randn(9, heads * vd + 3, generator=g)), C.bf16_round(1 + 0.2 * torch.randn(heads * vd, generator=g))
    zd = dev(z, dtype)
    got = B().head_gate_rms(o.cuda(), dev(w, dtype), zd[:, 3:], "silu", 1e-6, heads, vd, gate_first=True)
    gated = o.double() * R.silu(z[:, 3:].double())
    close(got, R.rms(gated.view(9, heads, vd), 1e-6).reshape(9, -1) * w.double(), dtype, tol16=2e-2)
    got = B().head_gate_rms(o.cuda(), dev(w, dtype), zd[:, 3:], "silu", 1e-6, heads, vd, gate_first=False)       # the other order differs
    close(got, R.rms(o.double().view(9, heads, vd), 1e-6).reshape(9, -1) * w.double() * R.silu(z[:, 3:].double()), dtype, tol16=2e-2)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,I", [(1024, 512), (1023, 520), (13109, 40), (700, 750)])
def test_many_gated_units_eight_values_to_a_thread(dtype, rows, I):
    # at, just above and below the 2^19 values from which a thread takes eight; 750 is no multiple of eight.  One stored rounding (2^-9 of
    # the value) plus a few fp32 ones
    g = torch.Generator().manual_seed(I)
    gu = C.bf16_round(torch.randn(rows, 2 * I, generator=g) * 2)
    d, gate, up = dev(gu, dtype), gu[:, :I].double(), gu[:, I:].double()
    silu = gate * torch.sigmoid(gate) * up
    close(B().silu_mul_rows(d), silu, dtype, tol32=2e-6, tol16=4e-3)
    close(B().glu_rows(d[:, :I], d[:, I:], "silu"), silu, dtype, tol32=2e-6, tol16=4e-3)
    ga = gate.clamp(max=1.25)
    close(B().clamp_glu_rows(d, 1.25), ga * torch.sigmoid(1.702 * ga) * (up.clamp(-1.25, 1.25) + 1), dtype, tol32=2e-6, tol16=4e-3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,d,top", [(256, 1028, 5), (255, 1028, 4), (300, 1026, 1), (300, 64, 8)])
def test_routed_sum_four_columns_to_a_thread(dtype, rows, d, top):
    g = torch.Generator().manual_seed(d + top)
    y, w = torch.randn(rows * top, d, generator=g), torch.rand(rows, top, generator=g)
    add, lg = C.bf16_round(torch.randn(rows, d, generator=g)), torch.randn(rows, generator=g)
    got = B().route_combine_gated(y.cuda(), w.cuda(), dev(add, dtype), lg.cuda(), DT[dtype])
    ref = torch.sigmoid(lg.double())[:, None] * add.double() + (w.double()[:, :, None] * y.double().view(rows, top, d)).sum(1)
    close(got, ref, dtype, tol32=2e-6, tol16=4e-3)                      # one stored rounding, top + 2 fp32 ones
    got = B().route_combine_pairs(y.cuda(), w.cuda(), torch.stack([y[:rows], y[-rows:]]).cuda(), None, DT[dtype])
    close(got, y[:rows].double() + y[-rows:].double() + (w.double()[:, :, None] * y.double().view(rows, top, d)).sum(1), dtype, tol32=2e-6, tol16=4e-3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,vd", [(3, 64), (2, 68), (3, 96), (5, 128), (2, 132), (4, 512), (2, 508), (3, 37)])
def test_norm_and_gate_of_heads_several_values_to_a_lane(dtype, heads, vd):
    g = torch.Generator().manual_seed(vd)
    n = heads * vd
    o, z, w = torch.randn(7, n, generator=g), C.bf16_round(torch.randn(7, n, generator=g)), C.bf16_round(1 + 0.2 * torch.randn(n, generator=g))
    zd, normed = dev(z, dtype), R.rms(o.double().view(7, heads, vd), 1e-6).reshape(7, -1)
    close(B().head_gate_rms(o.cuda(), dev(w, dtype), zd, "silu", 1e-6, heads, vd, gate_first=False), normed * w.double() * R.silu(z.double()),
          dtype, tol32=4e-6, tol16=4e-3)                                # one stored rounding, fp32 before it
    gated = (o.double() * R.silu(z.double())).view(7, heads, vd)
    close(B().head_gate_rms(o.cuda(), dev(w, dtype), zd, "silu", 1e-6, heads, vd, gate_first=True),
          R.rms(gated, 1e-6).reshape(7, -1) * w.double(), dtype, tol32=4e-6, tol16=4e-3)


@pytest.mark.parametrize("vd", [513, 516])
def test_norm_and_gate_of_wide_heads_beyond_a_grid(vd):
    # more heads than a launch's grid has, wider than the kernel of one wave per head holds: one value and four to an access
    heads = 65535 + 3
    g = torch.Generator(device="cuda").manual_seed(vd)
    o, z = (torch.randn(2, heads * vd, generator=g, device="cuda") for _ in range(2))
    w = 1 + 0.2 * torch.randn(vd, generator=g, device="cuda")
    for first in (True, False):
        got = B().head_gate_rms(o, w, z, "silu", 1e-6, heads, vd, gate_first=first).view(2, heads, vd)
        for h in (slice(0, 300), slice(heads - 300, heads)):      # both ends of the heads, in 64 bits
            a, act = o.view(2, heads, vd)[:, h].double().cpu(), R.silu(z.view(2, heads, vd)[:, h].double().cpu())
            ref = (R.rms(a * act, 1e-6) if first else R.rms(a, 1e-6) * act) * w.double().cpu()
            close(got[:, h].cpu(), ref, "float32", tol32=4e-6)    # as for the narrow heads above


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("channels,taps", [(301, 4), (514, 3), (513, 8), (1026, 5)])
def test_convolution_of_long_portions_in_walks_of_eight_rows(dtype, channels, taps):
    g = torch.Generator().manual_seed(channels)
    w, lens = C.bf16_round(torch.randn(channels, taps, generator=g)), (130, 5, 1, 77)      # entries end inside a walk of eight rows
    x = C.bf16_round(torch.randn(sum(lens), channels, generator=g))
    state = torch.randn(4, taps - 1, channels, generator=g)
    out = B().time_conv(dev(x, dtype), dev(w, dtype), state.cuda(), B().Ragged(list(lens), slots=[2, 0, 3, 1]), silu=True, out_dtype=torch.float32)
    at = 0
    for n, slot in zip(lens, (2, 0, 3, 1)):
        past = torch.cat([state[slot].double(), x[at:at + n].double()])
        ref = sum(past[j:j + n] * w[:, j].double() for j in range(taps))
        close(out[at:at + n], R.silu(ref), "float32", tol32=2e-6)
        at += n


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n", [7, 1 << 19, (1 << 19) + 5])
def test_squared_relu(dtype, n):
    x = C.bf16_round(torch.randn(n, generator=torch.Generator().manual_seed(n)))
    ref = torch.relu(x.double()) ** 2
    got = B().relu_sq(dev(x, dtype)).double().cpu()
    assert float(((got - ref).abs() - 2.0 ** -8 * ref).max()) <= 0       # at most one stored rounding


# ------------------------------------------------------------------ time convolution with biases
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("taps", [1, 2, 4, 7])
def test_time_convolution_with_input_and_output_bias_in_portions(dtype, taps):
    g = torch.Generator().manual_seed(taps)
    C_, lens = 70, [150, 9]
    u = [C.bf16_round(torch.randn(n, C_ + 4, generator=g)) for n in lens]
    w, ib, ob = (C.bf16_round(torch.randn(*s, generator=g) * 0.5) for s in ((C_, taps), (C_,), (C_,)))
    ref = [R.silu(R.tconv(x[:, 2:2 + C_].double() + ib.double(), w.double(), ob.double())) for x in u]
    for plan in ([[150, 9]], [[149, 1], [1, 8]], [[3, 2], [2, 1], [1, 1], [1, 1], [143, 4]]):
        state = torch.full((3, max(taps - 1, 1), C_), 7.0, device="cuda")       # slots 2 and 0 hold another request's tail
        state[[2, 0]] = 0.0
        outs, at = [[], []], [0, 0]
        for step in plan:
            rg = B().Ragged(step, slots=[2, 0])
            x = dev(torch.cat([u[i][at[i]:at[i] + n] for i, n in enumerate(step)]), dtype)
            o = B().time_conv(x[:, 2:], dev(w, dtype), state, rg, silu=True, out_dtype=torch.float32, channels=C_, in_bias=dev(ib, dtype),
                              out_bias=dev(ob, dtype))
            row = 0
            for i, n in enumerate(step):
                outs[i].append(o[row:row + n])
                at[i] += n
                row += n
        for i in range(2):
            close(torch.cat(outs[i]), ref[i], dtype, tol16=1e-2)
        assert float(state[1].min()) == 7.0                                      # a slot that is not in the step stays as it was


# ------------------------------------------------------------------ attention
class Paged:
    """one request's cache part over scattered pages, as a runtime lays it out: [k: slot, kv head, dim | v: slot, kv head, vdim]
    at offsets that do not start the page"""

    def __init__(self, page_ids, G, dim, dv, dtype, page_size=16):
        self.page_size = page_size
        self.k_off, self.v_off = 5 * 16, 5 * 16 + page_size * G * dim
        self.page_stride = self.v_off + page_size * G * dv + 3
        self.cache = torch.full(((max(page_ids) + 2) * self.page_stride,), float("nan"), dtype=DT[dtype], device="cuda")
        self.indptr = torch.tensor([0, len(page_ids)], dtype=torch.int32, device="cuda")
        self.pids = torch.tensor(page_ids, dtype=torch.int32, device="cuda")


PAGES = [7, 2, 11, 0, 5, 9, 3, 12, 1, 10, 4, 6, 8, 13, 14, 15, 16, 17, 18, 19]        # twenty pages of 16 tokens, in no order
# portions that end just before, at and just after page (16), window (21 / 40 / 70) and key tile (64) borders, then token by token
PORTIONS = [15, 1, 1, 6, 2, 23, 1, 1, 14, 2, 14] + [1] * 70


def dist_table(rel, bias_max):
    """the bias table expanded to one row per distance, as a runtime hands it to the attention"""
    rows = rel.shape[0]
    nd = 1
    while R.distance_bucket(nd - 1, rows, bias_max) < rows - 1:
        nd += 1
    return torch.stack([rel[R.distance_bucket(d, rows, bias_max)] for d in range(nd)]).float().cuda()


def run_conv_attention(m, w, p, h, dtype, plan, eps=1e-6):
    """the "attention" mixer as the runtime strings it together; plan: rows per step of ONE request"""
    Bk = B()
    H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    Wp = torch.cat([w[p + ".q"], w[p + ".k"], w[p + ".v"], w[p + ".g"]])
    ch = (H + G) * d + G * dv
    offs = [0, H * d, (H + G) * d]
    bias = torch.cat([w[p + ".q.b"], w[p + ".k.b"], w[p + ".v.b"]])
    pc = Paged(PAGES, G, d, dv, dtype)
    taps = m.get("conv", 0)
    state = torch.zeros((1, max(taps - 1, 1), ch), device="cuda")
    rot = m.get("rot")
    inv_freq = torch.tensor(R.rotation_frequencies(rot) if rot else [0.0], dtype=torch.float32).cuda()
    outs, at = [], 0
    for n in plan:
        rg = Bk.Ragged([n], starts=[at])
        proj = Bk.linear(dev(h[at:at + n], dtype), dev(Wp, dtype), plain=True)
        if taps:
            cw = torch.cat([w[p + ".q.conv"], w[p + ".k.conv"], w[p + ".v.conv"]])
            qkv = Bk.time_conv(proj, dev(cw, dtype), state, rg, out_dtype=torch.float32, channels=ch, in_bias=dev(bias, dtype))
            kw = {}
        else:
            qkv = proj
            kw = dict(q_bias=dev(w[p + ".q.b"], dtype), k_bias=dev(w[p + ".k.b"], dtype), v_bias=dev(w[p + ".v.b"], dtype))
        q = Bk.qk_prep_paged_form(qkv, offs, H, G, d, dv, rg, pc.indptr, pc.pids, pc.cache, pc.page_stride, pc.k_off, pc.v_off, 16,
                                  norm_kind="head_unit_after", eps=eps, inv_freq=inv_freq, rot_dims=rot["dims"] if rot else 0, halves=True, **kw)
        mix = Bk.paged_attention_masked(q, pc.cache, pc.page_stride, pc.k_off, pc.v_off, 16, rg, pc.indptr, pc.pids, G, dv, m["scale"],
                                        softcap=m.get("softcap", 0.0), gate=proj[:, ch:])
        outs.append(Bk.linear(mix, dev(w[p + ".o"], dtype), plain=True))
        at += n
    return torch.cat(outs)


def run_windowed_attention(m, w, p, h, dtype, plan, eps=1e-6, n_split=1):
    Bk = B()
    H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    Wp = torch.cat([w[p + ".q"], w[p + ".k"], w[p + ".v"], w[p + ".g"]])
    ch = (H + G) * d + G * dv
    offs = [0, H * d, (H + G) * d]
    pc = Paged(PAGES, G, d, dv, dtype)
    mk = m.get("mask") or {"size": 0, "keep_first": 0}
    tab = dist_table(w[p + ".rel"], m["bias_max"]) if m.get("bias_max") else None
    outs, at = [], 0
    for n in plan:
        rg = Bk.Ragged([n], starts=[at])
        proj = Bk.linear(dev(h[at:at + n], dtype), dev(Wp, dtype), plain=True)
        q = Bk.qk_prep_paged_form(proj, offs, H, G, d, dv, rg, pc.indptr, pc.pids, pc.cache, pc.page_stride, pc.k_off, pc.v_off, 16,
                                  q_norm=dev(w[p + ".q.norm"], dtype), k_norm=dev(w[p + ".k.norm"], dtype), norm_kind="all_weight", eps=eps,
                                  q_bias=dev(w[p + ".q.b"], dtype), k_bias=dev(w[p + ".k.b"], dtype), v_bias=dev(w[p + ".v.b"], dtype))
        mix = Bk.paged_attention_masked(q, pc.cache, pc.page_stride, pc.k_off, pc.v_off, 16, rg, pc.indptr, pc.pids, G, dv, m["scale"],
                                        window=mk["size"], keep_first=mk.get("keep_first", 0), dist_bias=tab, gate=proj[:, ch:],
                                        gate_per_head=True, n_split=n_split)
        outs.append(Bk.linear(mix, dev(w[p + ".o"], dtype), plain=True).float() + w[p + ".o.b"].cuda())
        at += n
    return torch.cat(outs)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layer", [("a", 1), ("a", 2), ("a", 4), ("wide", 0), ("odd", 0), ("b", 0), ("b", 2)])
def test_convolved_rotated_capped_attention_whole_and_in_portions(dtype, layer):
    cfg = C.CONFIGS[layer[0]]()
    w = C.random_weights(cfg, 4)
    p, m = "l%d.mix" % layer[1], cfg["layers"][layer[1]]["mixer"]
    n = 150
    h = C.bf16_round(torch.randn(n, cfg["width"], generator=torch.Generator().manual_seed(8)))
    ref = R.conv_attention(h.double(), w64(w), p, m, 1e-6)
    close(run_conv_attention(m, w, p, h, dtype, [n]), ref, dtype, tol32=1e-4, tol16=6e-2)
    close(run_conv_attention(m, w, p, h, dtype, PORTIONS), ref, dtype, tol32=1e-4, tol16=6e-2)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,H,G,d,dv,rot,kind", [(3, 5, 2, 66, 34, 66, "all_weight"), (520, 3, 1, 6, 10, 2, "head_weight"), (513, 6, 5, 128, 256, 64, "all_weight"),
                                                 (2, 9, 9, 256, 130, 256, "head_unit_after"), (2, 4, 1, 64, 3, 0, "head_weight")])
def test_heads_are_prepared_alike_one_or_two_values_to_a_lane(dtype, n, H, G, d, dv, rot, kind):
    """the same rows from an even column on (two values to a lane, unless a size is odd) and from an odd one, against float64"""
    Bk = B()
    g = torch.Generator().manual_seed(n + d)
    cols = (H + G) * d + G * dv
    x = C.bf16_round(torch.randn(n, cols, generator=g))
    bias = C.bf16_round(torch.randn(cols, generator=g))
    qn, kn = (H * d, G * d) if kind == "all_weight" else (d, d)
    qw, kw = C.bf16_round(1 + 0.2 * torch.randn(qn, generator=g)), C.bf16_round(1 + 0.2 * torch.randn(kn, generator=g))
    inv = torch.rand(max(rot // 2, 1), generator=g) / 4
    ang = torch.arange(n, dtype=torch.float64)[:, None, None] * inv.double()
    ref = (x + bias).double() if dtype == "float32" else (x.double() + bias.double())
    heads = []
    for t, w, k in ((ref[:, :H * d].view(n, H, d), qw, H), (ref[:, H * d:(H + G) * d].view(n, G, d), kw, G)):
        if kind == "all_weight":
            t = R.rms(t.reshape(n, -1), 1e-6).view(n, k, d) * w.double().view(k, d)
        elif kind == "head_weight":
            t = R.rms(t, 1e-6) * w.double()
        if rot:
            a, b = t[..., :rot // 2], t[..., rot // 2:rot]
            cs, sn = torch.cos(ang), torch.sin(ang)
            t = torch.cat([a * cs - b * sn, b * cs + a * sn, t[..., rot:]], -1)
        heads.append(R.rms(t, 1e-6) if kind == "head_unit_after" else t)
    rg = Bk.Ragged([n])
    for shift in (0, 1):
        pc = Paged(list(range((n + 15) // 16))[::-1], G, d, dv, dtype)
        pc.page_stride -= 1 - shift                   # the helper's pages are an odd number of values apart
        proj = torch.zeros(n, cols + 4, dtype=DT[dtype], device="cuda")
        proj[:, shift:shift + cols] = dev(x, dtype)
        b = dev(bias, dtype)
        q = Bk.qk_prep_paged_form(proj, [shift, shift + H * d, shift + (H + G) * d], H, G, d, dv, rg, pc.indptr, pc.pids, pc.cache, pc.page_stride,
                                  pc.k_off, pc.v_off, 16, q_norm=None if kind == "head_unit_after" else dev(qw, dtype),
                                  k_norm=None if kind == "head_unit_after" else dev(kw, dtype), norm_kind=kind, eps=1e-6, q_bias=b[:H * d],
                                  k_bias=b[H * d:(H + G) * d].clone(), v_bias=b[(H + G) * d:].clone(), inv_freq=inv.cuda(), rot_dims=rot, halves=True)
        close(q, heads[0], "float32", tol32=3e-5)     # fp32 angles up to 130 are off by 2^-24 of that: 8e-6 of a value
        flat = pc.cache.view(-1).double().cpu()
        page = pc.pids.cpu().long()
        rows = [(int(page[i // 16]) * pc.page_stride, i % 16) for i in range(n)]
        keys = torch.stack([flat[o + pc.k_off + sl * G * d:o + pc.k_off + (sl + 1) * G * d] for o, sl in rows])
        vals = torch.stack([flat[o + pc.v_off + sl * G * dv:o + pc.v_off + (sl + 1) * G * dv] for o, sl in rows])
        close(keys, heads[1].reshape(n, -1), dtype, tol32=3e-5, tol16=4e-3)
        close(vals, ref[:, (H + G) * d:], dtype, tol32=1e-6, tol16=4e-3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layer", [("a", 0), ("a", 3), ("wide", 1), ("odd", 1), ("odd", 2), ("b", 1)])
def test_windowed_biased_attention_whole_and_in_portions(dtype, layer):
    cfg = C.CONFIGS[layer[0]]()
    w = C.random_weights(cfg, 5)
    p, m = "l%d.mix.left" % layer[1], cfg["layers"][layer[1]]["mixer"]["left"]
    n = 150
    h = C.bf16_round(torch.randn(n, cfg["width"], generator=torch.Generator().manual_seed(9)))
    ref = R.windowed_attention(h.double(), w64(w), p, m, 1e-6)
    close(run_windowed_attention(m, w, p, h, dtype, [n]), ref, dtype, tol32=1e-4, tol16=6e-2)
    close(run_windowed_attention(m, w, p, h, dtype, PORTIONS), ref, dtype, tol32=1e-4, tol16=6e-2)
    close(run_windowed_attention(m, w, p, h, dtype, [100] + [1] * 50, n_split=5), ref, dtype, tol32=1e-4, tol16=6e-2)


def crafted_attention(dtype, n, plan, window=0, keep_first=0, softcap=0.0, tab=None, scale=1.0, hot=None, q_gain=1.0, n_split=1):
    """One head of 8 values whose queries and keys point along one axis: the key at `hot` is q_gain times longer, every value row
    carries its own position in its first column.  Returns what each row read from that column = the weighted mean position."""
    Bk = B()
    d = dv = 8
    q = torch.zeros(n, d)
    q[:, 0] = 1.0
    k = torch.zeros(n, d)
    k[:, 0] = 1.0
    if hot is not None:
        k[hot, 0] = q_gain
    v = torch.zeros(n, dv)
    v[:, 0] = torch.arange(n).float() / 64.0          # exact in bf16 up to 255 / 64... positions are told apart below by halves
    v[:, 1] = 1.0
    proj = dev(torch.cat([q, k, v], 1), dtype)
    pc = Paged(PAGES, 1, d, dv, dtype)
    outs, at = [], 0
    for m_ in plan:
        rg = Bk.Ragged([m_], starts=[at])
        qq = Bk.qk_prep_paged_form(proj[at:at + m_], [0, d, 2 * d], 1, 1, d, dv, rg, pc.indptr, pc.pids, pc.cache, pc.page_stride, pc.k_off,
                                   pc.v_off, 16)
        outs.append(Bk.paged_attention_masked(qq, pc.cache, pc.page_stride, pc.k_off, pc.v_off, 16, rg, pc.indptr, pc.pids, 1, dv, scale,
                                              softcap=softcap, window=window, keep_first=keep_first, dist_bias=tab, n_split=n_split))
        at += m_
    return torch.cat(outs).double().cpu()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("form", [{}, dict(window=40), dict(window=70, keep_first=10), dict(block=100)])
@pytest.mark.parametrize("shape", [(8, 2, 64, 64, 3), (6, 6, 20, 36, 1), (4, 1, 256, 256, 4), (8, 2, 72, 20, 2)])      # heads, kv heads, sizes, rows
def test_splits_without_a_key_leave_nothing_and_are_not_read(dtype, form, shape):
    """up to 64 workgroups share a row's keys: those past its last key tile (or past its window) end at once, whatever the workspace holds.  The
    sums differ from the unsplit launch's by their order alone (fp32), and by the rounding of weights against another maximum (bf16)."""
    Bk = B()
    H, G, d, dv, rows = shape
    gen = torch.Generator().manual_seed(d + rows)
    ps = 16 * G * (d + dv)
    cache = dev(torch.randn(70 * ps, generator=gen), dtype)
    ids, indptr = torch.randperm(70, generator=gen).int().cuda(), torch.tensor([0, 70], dtype=torch.int32).cuda()
    for start in (0, 61, 64, 500, 1100):
        rg = Bk.Ragged([rows], starts=[start])
        q = torch.randn(rows, H, d, generator=gen).cuda()
        call = lambda **kw: Bk.paged_attention_masked(q, cache, ps, 0, 16 * G * d, 16, rg, indptr, ids, G, dv, d ** -0.5, **form, **kw)  # noqa: E731
        whole = call()
        for n_split in (2, 16, 64):
            want = Bk.ffi.lib().pegainfer_paged_attention_workspace(Bk.attention_tiles(rg.lens, H // G, q.device)[0].numel(), G, dv, 1, n_split)
            poison = torch.full((want,), float("nan"), device="cuda")       # the block that the launch's workspace is taken from
            del poison
            close(call(n_split=n_split), whole.double().cpu(), dtype, tol32=2e-6, tol16=1e-2)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("plan", [[300], [290] + [1] * 10, [64, 64, 2, 62, 2, 96, 10]])
def test_one_far_key_among_hundreds_takes_the_weight(dtype, plan):
    """key 3 scores 30 against 1 for every other key: every later row reads (nearly) position 3, in a prompt's portion and in
    decoding, with the keys cut over workgroups or not"""
    for n_split in (1, 7):
        out = crafted_attention(dtype, 300, plan, hot=3, q_gain=30.0, n_split=n_split)
        assert float((out[10:, 0] * 64.0 - 3.0).abs().max()) < 1e-3 and float((out[:3, 0] * 64.0 - 3.0).abs().min()) > 0.5
    # the same key under a soft cap of 2: its score is held at 2 tanh(15), the others at 2 tanh(0.5): it no longer wins alone
    out = crafted_attention(dtype, 300, plan, hot=3, q_gain=30.0, softcap=2.0)
    e_hot, e_rest = math.exp(2.0 * math.tanh(15.0)), math.exp(2.0 * math.tanh(0.5))
    for i in (50, 299):
        want = (3 * e_hot + (i * (i + 1) / 2 - 3) * e_rest) / (e_hot + i * e_rest) / 64.0
        assert abs(float(out[i, 0]) - want) < (1e-5 if dtype == "float32" else 2e-2) * want


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("plan", [[200], [120] + [1] * 80, [60, 2, 2, 1, 1, 70, 64]])
@pytest.mark.parametrize("shape", [(21, 5), (64, 0), (70, 17), (3, 2), (16, 16)])
def test_marked_keys_at_the_window_edge_and_among_the_kept_first(dtype, plan, shape):
    """a key 30 times longer than the rest is seen exactly by the rows whose window holds it - or by all later rows when it is
    one of the kept first tokens"""
    size, keep = shape
    for hot in (max(keep - 1, 0), keep, keep + 40, 100):
        out = crafted_attention(dtype, 200, plan, window=size, keep_first=keep, hot=hot, q_gain=30.0)[:, 0] * 64.0
        for i in (hot, hot + 1, hot + size - 1, hot + size, hot + size + 1, 199):
            if i >= 200:
                continue
            seen = hot < keep or i - hot < size
            if seen:
                assert abs(float(out[i]) - hot) < 1e-2, (hot, i, float(out[i]))
            else:        # the row reads the mean position of what it does see (a bf16 output holds positions near 170 to +- 0.5)
                vis = [j for j in range(i + 1) if i - j < size or j < keep]
                assert abs(float(out[i]) - sum(vis) / len(vis)) < (1e-3 if dtype == "float32" else 1.01), (hot, i, float(out[i]))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_distance_bias_decides_the_softmax(dtype):
    """all keys alike; the bias table favours distance 9 by 25: every row reads the position 9 back (rows before 9: the mean of
    what they see); distances beyond the table's last row take that row"""
    tab = torch.zeros(12, 1)
    tab[9, 0] = 25.0
    for plan in ([100], [50] + [1] * 50):
        out = crafted_attention(dtype, 100, plan, tab=tab.cuda())[:, 0] * 64.0
        assert float((out[9:] - (torch.arange(9, 100).double() - 9)).abs().max()) < 1e-3
        assert abs(float(out[5]) - 2.5) < 1e-3
    tab = torch.zeros(12, 1)
    tab[11, 0] = 25.0               # every distance >= 11: the mean of positions 0 .. i - 11
    out = crafted_attention(dtype, 100, [100], tab=tab.cuda())[:, 0] * 64.0
    assert abs(float(out[99]) - 44.0) < (1e-3 if dtype == "float32" else 0.3) and abs(float(out[11]) - 0.0) < 1e-3


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_rotation_of_halves_with_given_frequencies_and_norm_after(dtype):
    g = torch.Generator().manual_seed(3)
    n, H, G, d, dv = 40, 3, 1, 14, 6
    rot = {"dims": 10, "base": 77.0, "scaling": {"factor": 5.0, "low": 1.0, "high": 3.0, "original": 30}}
    x = torch.randn(n, (H + G) * d + G * dv, generator=g)
    pc = Paged(PAGES, G, d, dv, dtype)
    rg = B().Ragged([n], starts=[100])           # a portion that starts at position 100
    inv_freq = torch.tensor(R.rotation_frequencies(rot), dtype=torch.float32).cuda()
    q = B().qk_prep_paged_form(x.cuda(), [0, H * d, (H + G) * d], H, G, d, dv, rg, pc.indptr, pc.pids, pc.cache, pc.page_stride, pc.k_off,
                               pc.v_off, 16, norm_kind="head_unit_after", eps=1e-6, inv_freq=inv_freq, rot_dims=10, halves=True)
    full = torch.zeros(140, H, d, dtype=F)
    full[100:] = x[:, :H * d].double().view(n, H, d)
    ref = R.rms(R.rotate_halves(full, rot), 1e-6)[100:]
    close(q, ref, "float32", tol32=3e-5)
    page, slot = PAGES[105 // 16], 105 % 16       # the key of position 105 sits in its page's slot
    kref = R.rms(R.rotate_halves(torch.cat([torch.zeros(100, G, d, dtype=F), x[:, H * d:(H + G) * d].double().view(n, G, d)]), rot), 1e-6)[105]
    got = pc.cache[page * pc.page_stride + pc.k_off + slot * G * d:][:G * d]
    close(got, kref.reshape(-1), dtype, tol32=3e-5, tol16=1e-2)


# ------------------------------------------------------------------ state-space scan
def run_state_space(m, w, p, h, dtype, plan, slots, state, conv_state, eps=1e-6):
    """the right half of "parallel" as the runtime strings it together; plan: steps of rows per entry; slots: entry -> state slot"""
    Bk = B()
    Hh, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    inner, ch = Hh * P, Hh * P + 2 * G * N
    outs, at = [[] for _ in h], [0] * len(h)
    for step in plan:
        live = [i for i, n in enumerate(step) if n]
        rg = Bk.Ragged([step[i] for i in live], slots=[slots[i] for i in live])
        x = dev(torch.cat([h[i][at[i]:at[i] + step[i]] for i in live]), dtype)
        proj = Bk.linear(x, dev(w[p + ".in"], dtype), plain=True)
        xbc = Bk.time_conv(proj[:, inner:], dev(w[p + ".conv"], dtype), conv_state, rg, silu=True, out_dtype=torch.float32, channels=ch,
                           out_bias=dev(w[p + ".conv.b"], dtype))
        y = Bk.ssd_scan(xbc, proj, inner + ch, dev(w[p + ".A_log"], dtype), dev(w[p + ".dt_bias"], dtype), dev(w[p + ".D"], dtype), state,
                        Hh, G, N, P, rg)
        ng = m.get("norm_groups", 1)
        mix = Bk.head_gate_rms(y, dev(w[p + ".norm"], dtype), proj, "silu", eps, ng, inner // ng, gate_first=True)
        o = Bk.linear(mix, dev(w[p + ".o"], dtype), plain=True)
        row = 0
        for i in live:
            outs[i].append(o[row:row + step[i]])
            at[i] += step[i]
            row += step[i]
    return [torch.cat(o) for o in outs]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layer", [("a", 0), ("a", 3), ("wide", 1), ("odd", 1), ("odd", 2), ("b", 1)])
def test_state_space_layer_whole_in_portions_and_in_dirty_slots(dtype, layer):
    cfg = C.CONFIGS[layer[0]]()
    w = C.random_weights(cfg, 6)
    p, m = "l%d.mix.right" % layer[1], cfg["layers"][layer[1]]["mixer"]["right"]
    g = torch.Generator().manual_seed(10)
    h = [C.bf16_round(torch.randn(n, cfg["width"], generator=g)) for n in (90, 37)]
    ref = [R.state_space(x.double(), w64(w), p, m, 1e-6) for x in h]
    floats = m["heads"] * m["state"] * m["vdim"]
    ch = m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
    for plan in ([[90, 37]], [[17, 1], [1, 1], [2, 2], [33, 0], [1, 33], [36, 0]], [[40, 30]] + [[1, 1]] * 7 + [[1, 0]] * 43):
        state = torch.full((4, floats), 3.0, device="cuda")              # slots 3 and 1 start from zero, the others hold strangers' state
        conv_state = torch.full((4, max(m["conv"] - 1, 1), ch), -2.0, device="cuda")
        state[[3, 1]] = 0.0
        conv_state[[3, 1]] = 0.0
        got = run_state_space(m, w, p, h, dtype, plan, [3, 1], state, conv_state)
        for i in range(2):
            close_rows(got[i], ref[i], dtype)
        assert float(state[0].min()) == 3.0 and float(state[2].max()) == 3.0


def test_an_old_write_is_kept_by_a_slow_head_and_forgotten_by_a_fast_one():
    """two heads read the same inputs; head 0 decays by exp(-0.001 dt), head 1 by exp(-20 dt).  Token 2 alone writes a large
    value: two hundred tokens later head 0 still reads it, head 1 reads nothing of it - in one step or token by token"""
    Bk = B()
    n, N, P = 260, 16, 8
    xbc = torch.zeros(n, 2 * P + 2 * N)
    xbc[:, 2 * P] = 1.0                      # B along the first state
    xbc[:, 2 * P + N] = 1.0                  # C along the first state
    xbc[2, :2 * P] = 50.0                    # the write
    proj = torch.zeros(n, 2)                 # raw step sizes 0: dt = softplus(0 + bias)
    A_log = torch.tensor([math.log(0.001), math.log(20.0)])
    dt_bias = torch.tensor([math.log(math.e - 1.0)] * 2)       # softplus -> 1
    D = torch.zeros(2)
    for plan in ([n], [10] + [1] * 250, [3, 1, 64, 64, 64, 64]):
        state = torch.zeros(1, 2 * N * P, device="cuda")
        ys, at = [], 0
        for m_ in plan:
            rg = Bk.Ragged([m_])
            ys.append(Bk.ssd_scan(xbc[at:at + m_].cuda(), proj[at:at + m_].cuda(), 0, A_log.cuda(), dt_bias.cuda(), D.cuda(), state, 2, 1, N, P, rg))
            at += m_
        y = torch.cat(ys).cpu()
        assert abs(float(y[202, 0]) - 50.0 * math.exp(-0.001 * 200)) < 1e-3 and abs(float(y[202, P])) < 1e-30
        assert abs(float(y[2, P]) - 50.0) < 1e-4 and float(y[1].abs().max()) == 0.0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,groups,N,P", [(4, 2, 128, 64), (2, 1, 16, 8), (3, 3, 20, 33), (2, 2, 256, 130), (1, 1, 5, 64)])
def test_state_space_chunks_against_the_scan_in_64_bits(dtype, heads, groups, N, P):
    """portions around the 64 tokens of a chunk beside one that stays with the scan, state left from an earlier portion, odd sizes and rows that are
    not aligned; heads that keep, fade and forget at once.  The scan in 64 bits is the reference: the outputs are sums of up to 320 products of
    about one, each a few 1e-6 off at most by the running product of the decays."""
    Bk = B()
    g = torch.Generator().manual_seed(N + P)
    lens, slots = [64, 3, 65, 320, 127], [1, 4, 0, 3, 5]
    inner = heads * P
    ch, T = inner + 2 * groups * N, sum(lens)
    xbc = torch.randn(T, ch, generator=g)
    xbc[:, inner:] *= N ** -0.25
    proj = C.bf16_round(torch.randn(T, heads + 3, generator=g))
    A_log = C.bf16_round(torch.tensor([[-9.0, -1.0, 3.0, 6.0][i % 4] for i in range(heads)]))
    dt_bias, D = C.bf16_round(torch.randn(heads, generator=g)), C.bf16_round(torch.randn(heads, generator=g))
    state = torch.randn(6, heads * N * P, generator=g).cuda()
    S = state.cpu().double().view(6, heads, N, P)
    rg = Bk.Ragged(lens, slots=slots)
    args = (dev(proj, dtype), 3, dev(A_log, dtype), dev(dt_bias, dtype), dev(D, dtype))
    y = Bk.ssd_scan(xbc.cuda(), *args, state, heads, groups, N, P, rg, scan_max=32).cpu().double()
    at = 0
    for n, s in zip(lens, slots):
        for h in range(heads):
            b0 = inner + (h // (heads // groups)) * N
            x, b, c = (xbc[at:at + n, k:k + w].double() for k, w in ((h * P, P), (b0, N), (b0 + groups * N, N)))
            dt = torch.nn.functional.softplus(proj[at:at + n, 3 + h].double() + dt_bias[h].double())
            a = torch.exp(-torch.exp(A_log[h].double()) * dt)
            St, ref = S[s, h].clone(), torch.empty(n, P, dtype=torch.float64)
            for t in range(n):
                St = a[t] * St + dt[t] * torch.outer(b[t], x[t])
                ref[t] = St.T @ c[t] + D[h].double() * x[t]
            tol = 2e-5 * max(1.0, float(ref.abs().max()))
            assert float((y[at:at + n, h * P:(h + 1) * P] - ref).abs().max()) < tol, (n, h)
            assert float((state[s].cpu().double().view(heads, N, P)[h] - St).abs().max()) < 2e-5 * max(1.0, float(St.abs().max())), (n, h)
        at += n
    assert torch.equal(state[2].cpu().double().view(heads, N, P), S[2])          # a slot of nobody


@pytest.mark.parametrize("N", [20, 5])
def test_state_space_chunks_keep_their_padding_zero(N):
    """state sizes that are no multiple of 16: an infinite value late in a chunk reaches no token of the blocks of 16 before its own"""
    Bk = B()
    g = torch.Generator().manual_seed(N)
    heads, P, T = 2, 33, 128
    inner = heads * P
    xbc, proj = torch.randn(T, inner + 2 * N, generator=g), torch.randn(T, heads, generator=g).cuda()
    xbc[60, 7] = float("inf")
    args = (proj, 0, torch.tensor([-1.0, 0.5]).cuda(), torch.randn(heads, generator=g).cuda(), torch.randn(heads, generator=g).cuda())
    y = Bk.ssd_scan(xbc.cuda(), *args, torch.ones(1, heads * N * P).cuda(), heads, 1, N, P, Bk.Ragged([T]), scan_max=32).cpu()
    assert torch.isfinite(y[:48]).all() and not torch.isfinite(y[60:, 7]).any()
    assert torch.isfinite(y[:, [i for i in range(inner) if i != 7]]).all()


@pytest.mark.parametrize("what", ["value", "key", "query", "step"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("N,P", [(128, 64), (20, 33), (5, 64)])
def test_state_space_chunks_let_nothing_reach_earlier_tokens(N, P, bad, what):
    """a value, key, query or step that is infinite or no number, at the start, inside and at the end of a block of 16 and of a chunk: exactly the
    outputs and states that the scan spoils are spoilt, the others stay within the rounding of sums of about a hundred products"""
    Bk = B()
    g = torch.Generator().manual_seed(N)
    heads, T = 2, 150
    inner, ch = heads * P, heads * P + 2 * N
    for at in (16, 45, 63, 64, 121):
        xbc, proj = torch.randn(T, ch, generator=g), torch.randn(T, heads, generator=g)
        xbc[:, inner:] *= N ** -0.25
        if what == "step":
            proj[at, 1] = bad
        else:
            xbc[at, {"value": P + P // 2, "key": inner + N - 1, "query": inner + N + 2}[what]] = bad
        args = (proj.cuda(), 0, torch.tensor([-1.0, 0.5]).cuda(), torch.randn(heads, generator=g).cuda(), torch.randn(heads, generator=g).cuda())
        runs = []
        for scan_max in (0, 32):
            state = torch.ones(1, heads * N * P).cuda()
            y = Bk.ssd_scan(xbc.cuda(), *args, state, heads, 1, N, P, Bk.Ragged([T]), scan_max=scan_max)
            runs += [y.cpu(), state.cpu()]
        for a, b in ((runs[0], runs[2]), (runs[1], runs[3])):
            ok = torch.isfinite(a)
            assert torch.equal(ok, torch.isfinite(b)), (at, int((ok != torch.isfinite(b)).sum()))
            assert float((a[ok] - b[ok]).abs().max()) < 1e-4 * max(1.0, float(a[ok].abs().max()))


def test_state_space_chunks_in_runs_of_bounded_scratch():
    """sizes whose scratch holds 31 chunks: runs that end inside an entry, at its last chunk and beyond, against the scan"""
    Bk = B()
    g = torch.Generator().manual_seed(3)
    heads, N, P, lens, slots = 16, 256, 512, [1900, 100, 2300, 20], [2, 0, 3, 1]
    T, inner = sum(lens), heads * P
    assert 2 ** 26 // Bk.ffi.lib().pegainfer_ssd_scan_workspace(1, heads, N, P) == 31
    xbc = torch.randn(T, inner + 2 * N, generator=g).cuda()
    xbc[:, inner:] *= N ** -0.25
    args = (torch.randn(T, heads, generator=g).cuda(), 0, torch.linspace(-4, 2, heads).cuda(), torch.randn(heads, generator=g).cuda(), torch.randn(heads, generator=g).cuda())
    runs = []
    for scan_max in (0, 64):
        state = torch.ones(4, heads * N * P).cuda()
        runs.append((Bk.ssd_scan(xbc, *args, state, heads, 1, N, P, Bk.Ragged(lens, slots=slots), scan_max=scan_max), state))
    for a, b in zip(*runs):
        assert float((a - b).abs().max()) < 2e-5 * float(a.abs().max())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("dim,vdim,off", [(128, 100, 0), (100, 128, 0), (24, 20, 0), (20, 24, 0), (24, 24, 4), (136, 130, 0), (40, 8, 0), (7, 64, 0)])
def test_general_attention_with_one_side_off_sixteen_bytes(dim, vdim, off, dtype):
    """a key or value size that is no multiple of eight, or values that start off 16 bytes, beside a side that is loaded in chunks: against the softmax
    in 64 bits; 1e-5 covers sums of 136 products and 90 weights in fp32, a bf16 output adds 2^-8 of it"""
    from pegainfer_amd import ops_blocks as B
    import ctypes
    g = torch.Generator().manual_seed(dim + vdim)
    H, G, page, lens, past = 4, 2, 16, [3, 70, 1], [0, 20, 65]
    T = sum(lens)
    need = [-(-(a + b) // page) for a, b in zip(lens, past)]
    v_off = -(-page * G * dim // 8) * 8 + off
    stride = -(-(v_off + page * G * vdim) // 8) * 8
    cache = torch.randn(sum(need) * stride, generator=g).to(DT[dtype])
    q = torch.randn(T, H, dim, generator=g)
    pos = [b + i for a, b in zip(lens, past) for i in range(a)]
    ent = [e for e, a in enumerate(lens) for _ in range(a)]
    first = np.cumsum([0] + need)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32).cuda()  # noqa: E731
    cd, qd, posd, entd, ind, ids = cache.cuda(), q.cuda(), i32(pos), i32(ent), i32(first.tolist()), i32(list(range(sum(need))))
    t = B.attention_tiles(lens, H // G, "cuda", 16)
    out = torch.full((T, H * vdim), float("nan"), dtype=DT[dtype], device="cuda")
    a = B.AttnOptions(n_split=1, plain=1)
    B._chk(B.ffi.lib().pegainfer_paged_attention_opt(
        qd.data_ptr(), cd.data_ptr(), stride, 0, v_off, page, posd.data_ptr(), entd.data_ptr(), ind.data_ptr(), ids.data_ptr(), H, G, dim, vdim,
        dim ** -0.5, 1.0, *(c.data_ptr() for c in t), t[0].numel(), out.data_ptr(), out.stride(0), ctypes.addressof(a), B._dt(cd), B._stream()), "attention")
    pages = cache.double().view(-1, stride)
    for r in range(T):
        mine = pages[first[ent[r]]:first[ent[r] + 1]]
        k = mine[:, :page * G * dim].reshape(-1, G, dim)[:pos[r] + 1]
        v = mine[:, v_off:v_off + page * G * vdim].reshape(-1, G, vdim)[:pos[r] + 1]
        for h in range(H):
            ref = torch.softmax(k[:, h // 2] @ q[r, h].double() * dim ** -0.5, 0) @ v[:, h // 2]
            got = out[r, h * vdim:(h + 1) * vdim].cpu().double()
            assert ((got - ref).abs() <= 1e-5 + (ref.abs() / 256 if dtype == "bfloat16" else 0)).all(), (r, h)


@pytest.mark.parametrize("tile_rows", [32, 64])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("H,G,dim,window", [(4, 4, 64, 0), (8, 2, 128, 0), (8, 2, 256, 0), (4, 4, 128, 20)])
def test_wide_tiles_bring_no_value_further_than_sixteen_rows(H, G, dim, window, bad, tile_rows):
    """a value that is infinite or no number reaches, beside the rows that see it, at most those that share sixteen rows with one of them (as in the
    form of 16-row tiles), not the rest of a wide tile: the others are bit for bit what they are without it"""
    from pegainfer_amd import ops_blocks as B
    import ctypes
    g = torch.Generator().manual_seed(dim)
    page, T, per = 16, 100, H // G
    need = -(-T // page)
    stride = page * G * 2 * dim
    v_off = page * G * dim
    sound = torch.randn(need * stride, generator=g).bfloat16()
    qd = torch.randn(T, H, dim, generator=g).cuda()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32).cuda()  # noqa: E731
    pos, ent, ind, ids = i32(list(range(T))), i32([0] * T), i32([0, need]), i32(list(range(need)))
    t = B.attention_tiles([T], per, "cuda", tile_rows)

    def run(cache):
        cd, out = cache.cuda(), torch.empty(T, H * dim, dtype=torch.bfloat16, device="cuda")
        a = B.AttnOptions(n_split=1, tile_rows=tile_rows, window=window)
        B._chk(B.ffi.lib().pegainfer_paged_attention_opt(
            qd.data_ptr(), cd.data_ptr(), stride, 0, v_off, page, pos.data_ptr(), ent.data_ptr(), ind.data_ptr(), ids.data_ptr(), H, G, dim, dim,
            dim ** -0.5, 1.0, *(c.data_ptr() for c in t), t[0].numel(), out.data_ptr(), out.stride(0), ctypes.addressof(a), 0, B._stream()), "attention")
        return out.cpu()

    ref = run(sound)
    for at in (0, 15, 31, 40, 63, 64, 99):
        cache = sound.clone()
        cache.view(need, stride)[at // page, v_off + (at % page) * G * dim + 3] = bad          # head 0 of that token
        got = run(cache)
        group, per_tile = 16 // per, tile_rows // per            # tokens of sixteen rows, of a tile
        sees = [at <= r and (not window or r - at < window) for r in range(T)]
        first = lambda r: r // per_tile * per_tile + r % per_tile // group * group  # noqa: E731
        near = {first(r) for r in range(T) if sees[r]}
        for r in range(T):
            if sees[r]:
                assert not torch.isfinite(got[r, 3]), (at, r)
            elif first(r) not in near:
                assert torch.equal(got[r], ref[r]), (at, r)


FORMS = {"plain": {}, "cap far above the scores": {"softcap": 60.0}, "binding cap": {"softcap": 1.5}, "window and kept first": {"window": 37, "keep_first": 3},
         "table bias": {"bias": 90, "window": 150}, "slope and cap": {"slope": True, "softcap": 4.0}, "blocks and sink": {"block": 48, "sink": True},
         "gate per value, head norm": {"gate": 1, "norm": True}, "gate per head, bias": {"gate": 2, "bias": 20}}


@pytest.mark.parametrize("tile_rows", [32, 64])
@pytest.mark.parametrize("dim,vdim,page", [(24, 40, 16), (64, 64, 8), (72, 128, 5), (128, 128, 16), (136, 256, 32), (256, 72, 16)])
@pytest.mark.parametrize("form", FORMS)
def test_wide_tiles_take_every_form(form, dim, vdim, page, tile_rows):
    """The kernel for prompts against the fp32-FMA kernel on the same bf16 cache: every option, rows of one and two halves of 256 bytes and more,
    rows whose last chunks are padding, pages that hold a whole number of a DMA's rows and pages that do not, entries that end around a
    64-key tile, a portion behind a cached prefix.  The matrix cores see q and the weights in bf16 (2^-9 each, relative); a score of size s moves by
    2^-9 s and with it its weight: 2^-7 of the largest value covers s up to 4 at these scales."""
    from pegainfer_amd import ops_blocks as B
    import ctypes
    o = FORMS[form]
    g = torch.Generator().manual_seed(dim * 7 + vdim + page)
    H, G = 6, 2
    lens, past = [1, 63, 64, 65, 130, 7], [0, 0, 0, 3, 0, 140]
    T = sum(lens)
    need = [-(-(a + b) // page) for a, b in zip(lens, past)]
    order = torch.randperm(sum(need), generator=g).int()
    indptr = torch.tensor([0] + np.cumsum(need).tolist(), dtype=torch.int32)
    stride = (page * G * (dim + vdim) + 7) // 8 * 8
    v_off = page * G * dim
    cache = torch.randn(sum(need) * stride, generator=g).bfloat16().cuda()
    q = torch.randn(T, H, dim, generator=g).cuda()
    pos = torch.cat([torch.arange(b, a + b) for a, b in zip(lens, past)]).int().cuda()
    ent = torch.cat([torch.full((a,), i) for i, a in enumerate(lens)]).int().cuda()
    ind, ids = indptr.cuda(), order.cuda()
    sink, bias = torch.randn(H, generator=g).bfloat16().cuda(), torch.randn(max(1, o.get("bias", 1)), H, generator=g).cuda()
    slope, gate = torch.rand(H, generator=g).cuda() * 0.1, torch.randn(T, H * vdim, generator=g).bfloat16().cuda()
    outs = []
    for rows, plain in ((16, 1), (tile_rows, 0)):
        t = B.attention_tiles(lens, H // G, "cuda", rows)
        out = torch.full((T, H * vdim), float("nan"), dtype=torch.bfloat16, device="cuda")
        a = B.AttnOptions(softcap=o.get("softcap", 0.0), window=o.get("window", 0), keep_first=o.get("keep_first", 0), block=o.get("block", 0),
                          dist_bias=bias.data_ptr() if "bias" in o else None, n_dist=o.get("bias", 0), dist_slope=slope.data_ptr() if "slope" in o else None,
                          sink=sink.data_ptr() if "sink" in o else None, head_norm=int(o.get("norm", False)), norm_eps=1e-6,
                          gate=gate.data_ptr() if "gate" in o else None, gate_stride=H * vdim, gate_kind=o.get("gate", 0), n_split=1, plain=plain,
                          tile_rows=rows if rows > 16 else 0)
        B._chk(B.ffi.lib().pegainfer_paged_attention_opt(
            q.data_ptr(), cache.data_ptr(), stride, 0, v_off, page, pos.data_ptr(), ent.data_ptr(), ind.data_ptr(), ids.data_ptr(), H, G, dim, vdim,
            dim ** -0.5, 1.0, *(c.data_ptr() for c in t), t[0].numel(), out.data_ptr(), out.stride(0), ctypes.addressof(a), 0, B._stream()), "attention")
        outs.append(out.float().cpu())
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -7 * outs[0].abs().max()
