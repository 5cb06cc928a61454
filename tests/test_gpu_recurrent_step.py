"""One launch per decode step of the recurrences with a matrix state per head, against float64: sizes at and off the launch's own (rows of the
state in sixteens, columns in fours), grouped keys, second-stage projections on the way or beforehand, several steps through one state."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def rounded(*shape, g, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).bfloat16().float()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["gated", "delta", "delta_channel"])
@pytest.mark.parametrize("n,heads,kv,dim,vdim,rank,on_the_way", [(3, 4, 4, 128, 128, 16, True), (1, 6, 3, 16, 4, 5, True), (5, 2, 1, 100, 68, 40, False),
                                                               (2, 3, 3, 1, 64, 8, True), (9, 2, 2, 33, 124, 72, True)])
def test_step_against_float64(dtype, kind, n, heads, kv, dim, vdim, rank, on_the_way):
    from pegainfer_amd import ops_blocks as B
    if kind == "gated":
        kv = heads
    g = torch.Generator().manual_seed(dim * 3 + vdim)
    dt, dev = DT[dtype], lambda t: t.to(DT[dtype]).cuda().contiguous()
    qk, vals, pad = kv * dim, heads * vdim, -(-rank // 8) * 8
    low, glow, a_off, b_off, g_off, width = 0, pad, 2 * pad, 2 * pad + heads, 2 * pad + 2 * heads, 2 * pad + 2 * heads + vals
    width = -(-width // 8) * 8
    offs_x = [0, qk, 2 * qk]
    x_width = -(-(2 * qk + vals) // 4) * 4
    offs = [o if kind != "gated" else -(-width // 8) * 8 + o for o in offs_x]
    if offs[2] % 4:                                # the launch reads values in fours
        offs[2] += 4 - offs[2] % 4
        x_width += 4
    w_up, w_gate = rounded(heads * dim, rank, g=g, scale=rank ** -0.5), rounded(vals, rank, g=g, scale=rank ** -0.5)
    z_bias = rounded(heads if kind == "delta" else heads * dim, g=g)
    A_log, norm_w = rounded(heads, g=g, scale=0.3), rounded(vdim, g=g, scale=0.2) + 1
    slots = torch.randperm(n + 2, generator=g)[:n].to(torch.int32)
    state = torch.randn(n + 2, heads * dim * vdim + 4, generator=g)
    S = state[slots.long(), :heads * dim * vdim].double().view(n, heads, dim, vdim)
    st = state.cuda()
    padded = lambda w: torch.cat([w, torch.zeros(w.shape[0], pad - rank)], 1)
    for step in range(3):
        rows = rounded(n, width, g=g)
        x = rounded(n, x_width, g=g) if kind == "gated" else torch.randn(n, x_width, generator=g)
        full = torch.cat([rows, x], 1) if kind == "gated" else rows
        if full.shape[1] % 8:
            full = torch.cat([full, torch.zeros(n, 8 - full.shape[1] % 8)], 1)
        off0 = width if kind == "gated" else 0
        q = x[:, offs[0] - off0:][:, :qk].double().view(n, kv, dim).repeat_interleave(heads // kv, 1)
        k = x[:, offs[1] - off0:][:, :qk].double().view(n, kv, dim).repeat_interleave(heads // kv, 1)
        v = x[:, offs[2] - off0:][:, :vals].double().view(n, heads, vdim)
        r64 = rows.double()
        z = r64[:, low:low + rank] @ w_up.double().T
        if kind == "gated":
            a = torch.sigmoid(z + z_bias.double()).pow(1 / 4.0).view(n, heads, dim, 1)
            S = a * S + k[..., None] * v[:, :, None]
            y = (S * q[..., None]).sum(2) * dim ** -0.5
        else:
            q, k = (t / (t.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt() for t in (q, k))
            soft = torch.nn.functional.softplus
            if kind == "delta":
                a = torch.exp(-A_log.double().exp() * soft(r64[:, a_off:a_off + heads] + z_bias.double())).view(n, heads, 1, 1)
            else:
                a = torch.exp(-A_log.double().exp().repeat_interleave(dim) * soft(z + z_bias.double())).view(n, heads, dim, 1)
            beta = torch.sigmoid(r64[:, b_off:b_off + heads]).view(n, heads, 1)
            S = a * S
            S = S + k[..., None] * (beta * (v - (S * k[..., None]).sum(2)))[:, :, None]
            y = (S * q[..., None]).sum(2) * dim ** -0.5
        gz = r64[:, glow:glow + rank] @ w_gate.double().T if on_the_way else r64[:, g_off:g_off + vals]
        if on_the_way:
            gz = gz.to(torch.float32).to(dt).double()
        gate = torch.sigmoid(gz) if kind == "delta_channel" else gz * torch.sigmoid(gz)
        ref = (y / (y.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt() * norm_w.double()).reshape(n, -1) * gate * 0.5
        d_rows, z32 = dev(full), z.float().cuda()
        got = B.recurrent_step(kind, d_rows if kind == "gated" else x.cuda(), offs, d_rows, st, slots.cuda(), dev(norm_w), heads, kv, dim, vdim,
                               q_scale=dim ** -0.5, z=None if on_the_way else z32, w_up=dev(padded(w_up)) if on_the_way else None, low_off=low,
                               rank=rank, z_bias=dev(z_bias), tau=4.0, A_log=dev(A_log), a_off=a_off, b_off=b_off,
                               gate=None if on_the_way else d_rows[:, g_off:], w_gate=dev(padded(w_gate)) if on_the_way else None, gate_low_off=glow,
                               gate_rank=rank, gate_kind="sigmoid" if kind == "delta_channel" else "silu", factor=0.5)
        # fp32 throughout, then one stored rounding (2^-9) of the row and one of a gate made on the way, which may fall on the other side of a tie
        err = float((got.double().cpu() - ref).abs().max() / ref.abs().max())
        assert err < (2e-5 if dtype == "float32" else 8e-3), (step, err)
        flat = st[slots.long().cuda(), :heads * dim * vdim].double().cpu().view(S.shape)
        err = float((flat - S).abs().max() / S.abs().max())
        assert err < 1e-5, (step, err)
    untouched = [i for i in range(n + 2) if i not in slots.tolist()]
    assert torch.equal(st[untouched].cpu(), state[untouched])


def test_sizes_that_the_launch_leaves_to_the_others():
    from pegainfer_amd import ops_blocks as B
    for dim, vdim in ((129, 64), (64, 132), (64, 66)):
        proj, slots = torch.zeros(1, 2 * dim + vdim + 8, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
        assert B.recurrent_step("gated", proj, [0, dim, 2 * dim], proj, torch.zeros(1, dim * vdim, device="cuda"), slots, torch.ones(vdim, device="cuda"),
                                1, 1, dim, vdim, z=torch.zeros(1, dim, device="cuda"), gate=proj) is None


# the scan behind them: rounds of sixteen tokens (edges, remainders, an empty entry), values in fours and one by one, every number of values a lane holds
@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("heads,kv,dim,vdim,lens", [(2, 1, 16, 16, [1, 15, 16]), (2, 2, 30, 20, [17, 2]), (2, 1, 64, 33, [0, 33, 1]), (1, 1, 100, 16, [48]),
                                                    (4, 2, 128, 48, [31, 3, 16]), (2, 2, 99, 30, [32, 5]), (1, 1, 200, 17, [18])])
@pytest.mark.parametrize("odd", [False, True])
def test_delta_scan_against_float64(channel, heads, kv, dim, vdim, lens, odd):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(dim + vdim)
    n, width = sum(lens), 2 * kv * dim + heads * vdim
    qkv = torch.randn(n, width + (4 - width % 4) % 4 + int(odd), generator=g)
    proj, a = torch.randn(n, 2 * heads, generator=g), torch.randn(n, heads * dim, generator=g)
    A_log, dt_bias = torch.randn(heads, generator=g) * 0.3, torch.randn(heads * (dim if channel else 1), generator=g)
    state = torch.randn(len(lens) + 1, heads, dim, vdim, generator=g)
    slots = torch.randperm(len(lens) + 1, generator=g)[:len(lens)].tolist()
    unit = lambda t: t / (t.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()
    parts = lambda o: qkv[:, o:o + kv * dim].double().view(n, kv, dim).repeat_interleave(heads // kv, 1)
    q, k = unit(parts(0)) * dim ** -0.5, unit(parts(kv * dim))
    v, beta = qkv[:, 2 * kv * dim:width].double().view(n, heads, vdim), torch.sigmoid(proj[:, :heads].double())
    z = a.double() if channel else proj[:, heads:].double()
    rate = A_log.double().exp().repeat_interleave(dim) if channel else A_log.double().exp()
    decay = torch.exp(-rate * torch.nn.functional.softplus(z + dt_bias.double())).view(n, heads, -1, 1)
    want, at, after = torch.zeros(n, heads, vdim, dtype=torch.float64), 0, state.double().clone()
    for length, slot in zip(lens, slots):
        S = after[slot]
        for t in range(at, at + length):
            S = decay[t] * S
            S = S + k[t][..., None] * (beta[t][:, None] * (v[t] - (S * k[t][..., None]).sum(1)))[:, None]
            want[t] = (S * q[t][..., None]).sum(1)
        after[slot], at = S, at + length
    rg, mem, x = B.Ragged(lens, slots), state.cuda(), qkv.cuda()
    if channel:
        o = B.delta_rule_channel(x, proj.cuda(), 0, a.cuda(), A_log.cuda(), dt_bias.cuda(), mem, heads, kv, dim, vdim, rg)
    else:
        o = B.delta_rule(x, proj.cuda(), 0, heads, A_log.cuda(), dt_bias.cuda(), mem, heads, kv, dim, vdim, rg)
    # at most 48 steps of fp32 sums of at most 200 terms, each a contraction: some 1e-6 of the largest value; five times that is asked for
    assert float((o.double().cpu().view(n, heads, vdim) - want).abs().max() / want.abs().max()) < 5e-6
    assert float((mem.double().cpu() - after).abs().max() / after.abs().max()) < 5e-6
