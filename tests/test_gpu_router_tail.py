"""The router behind a row (decode steps): logits, selection and gate logit in the launch that leaves the row, and the experts' products that find
their rows from the choices.  Against double precision on the stored rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SIGMOID, SOFTMAX, TOP2, MAX = 0, 1, 0, 1


def select(z, corr, G, keep, top, score, group_kind, renorm, factor):
    """the selection by itself, one row of logits in double precision"""
    s = torch.sigmoid(z) if score == SIGMOID else torch.softmax(z, -1)
    ch = s + corr if corr is not None else s.clone()
    E = z.numel()
    if G > 1:
        per = E // G
        best = ch.view(G, per).sort(-1, descending=True).values
        gs = best[:, :2].sum(-1) if per >= 2 and group_kind == TOP2 else best[:, 0]
        dropped = gs.argsort(descending=True, stable=True)[keep:]
        ch.view(G, per)[dropped] = -float("inf")
    idx = ch.argsort(descending=True, stable=True)[:top]
    found = torch.isfinite(ch[idx])
    w = torch.where(found, s[idx], torch.zeros((), dtype=s.dtype))
    idx = torch.where(found, idx, torch.zeros_like(idx))
    return idx, w * factor / ((w.sum() + 1e-20) if renorm else 1.0)


@pytest.mark.parametrize("kind", ["join", "scalar", "group", "dyt"])
@pytest.mark.parametrize("rows,d,E,gate,G,keep,top,score,group_kind,renorm", [
    (1, 32, 1, 0, 1, 1, 1, SIGMOID, TOP2, 0), (3, 1024, 16, 1, 4, 2, 4, SOFTMAX, MAX, 1), (2, 1056, 17, 0, 1, 1, 3, SIGMOID, TOP2, 1),
    (16, 2048, 47, 1, 1, 1, 8, SOFTMAX, MAX, 0), (5, 2560, 32, 0, 4, 1, 9, SOFTMAX, TOP2, 0), (4, 4096, 48, 0, 8, 4, 6, SIGMOID, TOP2, 0)])
def test_a_row_is_routed_by_the_launch_that_leaves_it(kind, rows, d, E, gate, G, keep, top, score, group_kind, renorm):
    """widths of one piece and at the thread counts' edges, one to three blocks of experts, more choices than eligible experts.  A logit is a
    fp32 sum of d exact products of about 1 / sqrt(d) times one: 1e-6 sqrt(d) at most; weights follow within twice that."""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(rows * 10000 + d + E)
    bf = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    w = (torch.randn(E + gate, d, generator=g) * 3 / d ** 0.5).bfloat16().cuda()
    corr = (torch.randn(E, generator=g) * 0.1).bfloat16().cuda() if score == SIGMOID else None
    oe, ow = torch.full((rows, top), -1, dtype=torch.int32, device="cuda"), torch.full((rows, top), float("nan"), device="cuda")
    gl = torch.full((rows, 3), float("nan"), device="cuda")
    t = B.RouterTailDesc(w=w.data_ptr(), correction=None if corr is None else corr.data_ptr(), out_expert=oe.data_ptr(), out_weight=ow.data_ptr(),
                         gate_logit=gl.data_ptr() + 4 if gate else None, gate_stride=3, experts=E, n_groups=G, keep_groups=keep, top=top, score_kind=score,
                         group_kind=group_kind, renorm=renorm, factor=1.5)
    x0, y = torch.randn(rows, d, generator=g).cuda(), bf(rows, d)

    def launch(router):
        x = x0.clone()
        if kind == "join":
            row = B.join_rms(x, bf_post, gain=bf_gain, y=y, router=router)
        elif kind == "dyt":
            row = torch.zeros(rows, d, dtype=torch.bfloat16, device="cuda")
            B.dyt_step(torch.bfloat16, rows, d, x=x, y=y, post_alpha=one, post_w=bf_post, post_b=bf_gain, next_alpha=one, next_w=bf_gain,
                       next_b=bf_post, out=row, router=router)
        else:
            row, st = torch.zeros(rows, d, dtype=torch.bfloat16, device="cuda"), state.clone()
            form = dict(groups=1, xb_out=row) if kind == "group" else dict(conv_w=taps, conv_state=st, conv_slot_stride=3 * d, conv_slot=slot, conv_out=row)
            B.row_step(torch.bfloat16, rows, d, x_in=x, x_out=x, y=y, mult=0.7, gain=bf_gain, eps=1e-5, router=router, **form)
        return row, x
    bf_post, bf_gain, one = bf(d), bf(d), torch.ones(1, dtype=torch.bfloat16, device="cuda")
    state, taps, slot = torch.randn(rows, 3 * d, generator=g).cuda(), bf(d, 4), torch.arange(rows, dtype=torch.int32, device="cuda")
    row, x = launch(t)
    plain, xp = launch(None)
    # the same row and stream as without a router (another number of threads may sum a norm in another order: an ulp of bf16, a few of fp32)
    assert float((row.double() - plain.double()).abs().max()) <= 2.0 ** -7 * float(plain.double().abs().max())
    assert torch.allclose(x, xp, rtol=1e-6, atol=1e-6)
    z = (row.double() @ w.double().T).cpu()
    tol = 1e-6 * d ** 0.5 * float(1 + z.abs().max())
    if gate:
        assert float((gl[:, 1].double().cpu() - z[:, E]).abs().max()) < tol and bool(gl[:, 0].isnan().all())
    for r in range(rows):
        idx, wt = select(z[r, :E], None if corr is None else corr.double().cpu(), G, keep, top, score, group_kind, renorm, 1.5)
        assert oe[r].tolist() == idx.tolist(), (r, oe[r].tolist(), idx.tolist())
        assert float((ow[r].double().cpu() - wt).abs().max()) < 4 * tol


@pytest.mark.parametrize("rows,d,E,gate,dtype", [(1, 1000, 8, 0, 0), (1, 4128, 8, 0, 0), (1, 1024, 48, 1, 0), (1, 1024, 49, 0, 0), (1, 1024, 8, 0, 1)])
def test_other_routers_stay_launches_of_their_own(rows, d, E, gate, dtype):
    from pegainfer_amd import ffi
    from pegainfer_amd import ops_blocks as B
    assert not ffi.lib().pegainfer_router_tail_ok(E, gate, d, dtype)
    dt = torch.float32 if dtype else torch.bfloat16
    x, row, w = torch.zeros(rows, d, device="cuda"), torch.zeros(rows, d, dtype=dt, device="cuda"), torch.zeros(E + gate, d, dtype=dt, device="cuda")
    v, oe, ow = torch.zeros(d, dtype=dt, device="cuda"), torch.zeros(rows, 2, dtype=torch.int32, device="cuda"), torch.zeros(rows, 2, device="cuda")
    t = B.RouterTailDesc(w=w.data_ptr(), out_expert=oe.data_ptr(), out_weight=ow.data_ptr(), gate_logit=ow.data_ptr() if gate else None, experts=E,
                         n_groups=1, keep_groups=1, top=2, score_kind=SOFTMAX, factor=1.0)
    with pytest.raises(RuntimeError):
        B.join_rms(x, v, gain=v, y=row, router=t)


def test_large_routers_are_left_to_a_product_of_their_own():
    from pegainfer_amd import ffi
    ok = lambda E, gate, d: ffi.lib().pegainfer_router_tail_ok(E, gate, d, 0)  # noqa: E731
    assert ok(48, 0, 2560) and ok(47, 1, 2560) and not ok(48, 0, 2592) and ok(30, 0, 4096) and not ok(30, 1, 4096)


@pytest.mark.parametrize("T,top,E,kind", [(1, 1, 1, "even"), (3, 4, 5, "even"), (16, 4, 64, "even"), (16, 16, 33, "even"), (16, 4, 7, "first"),
                                          (13, 5, 9, "beyond"), (2, 3, 6, "none")])
@pytest.mark.parametrize("glu,slices,found", [(0, 0, False), (1, 2, False), (1, 1, True)])
def test_experts_find_their_rows_from_the_choices(T, top, E, kind, glu, slices, found):
    """one to 256 pairs, experts with more than one tile (rows whose choices all fall on expert 0), choices beyond the experts (no rows), none at
    all: each pair's row through both products, bit for bit what the table's form gives; rows without an expert stay as they were"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(T * 100 + top + E)
    ff, D, two = 40, 72, 2 if glu else 1
    sff = slices * ff
    bf = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    x, up, down, s_up, s_down = bf(T, D), bf(E, two * ff, D), bf(E, D, ff), bf(max(1, two * sff), D), bf(D, max(1, sff))
    if kind == "first":
        expert = torch.zeros(T, top, dtype=torch.int32)
    elif kind == "none":
        expert = torch.full((T, top), E, dtype=torch.int32)
    else:
        most = E + 3 if kind == "beyond" else E
        expert = torch.stack([torch.randperm(max(most, top), generator=g)[:top] % most for _ in range(T)]).int()
    e = expert.cuda()
    P, n = T * top, T * top + slices * T
    shared = dict(shared_groups=slices, shared_rows=T, shared_pos0=P)

    def both(chosen):
        act, y = torch.full((n, ff), 7.0, device="cuda").bfloat16(), torch.full((n, D), 7.0, device="cuda")
        table1 = table2 = {}
        if not chosen:
            pp, pr, tg, t0, tr, nt, mt = B.route_sort(e, E)
            hold.extend([pp, pr, tg, t0, tr, nt])
            table1 = dict(tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(), max_tiles=mt, max_tile_rows=16,
                          tile_rows_cap=64, x_row_index=pr.data_ptr(), y_row_index=pp.data_ptr())
            table2 = dict(table1, x_row_index=pp.data_ptr())
        a = dict(choices=e, experts=E, tiles=torch.full((B.CHOSEN_WORDS,), 1 << 30, dtype=torch.int32, device="cuda") if found else None) if chosen else {}
        g1 = B.GemmDesc(x=x.data_ptr(), w=up.data_ptr(), y=act.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=0, m=ff, k=D, x_row_stride=D, w_m_stride=D,
                        w_k_stride=1, w_group_stride=two * ff * D, y_row_stride=ff, epilogue=0 if glu else B.EPI_RELU_SQ, **table1)
        B.expert_rows(B.ExpertRowsDesc(g=g1, glu=glu, shared_w=s_up.data_ptr() if slices else None, shared_m_stride=D, shared_group_stride=ff * D,
                                       shared_up=sff * D, **shared), **a)
        g2 = B.GemmDesc(x=act.data_ptr(), w=down.data_ptr(), y=y.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=1, m=D, k=ff, x_row_stride=ff, w_m_stride=ff,
                        w_k_stride=1, w_group_stride=D * ff, y_row_stride=D, **table2)
        if chosen or not slices:
            B.expert_rows(B.ExpertRowsDesc(g=g2, shared_w=s_down.data_ptr() if slices else None, shared_m_stride=sff, shared_group_stride=ff, **shared),
                          **dict(a, by_pair=True) if chosen else {})
        return act, y
    hold = []
    act, y = both(True)
    a64 = act.double().cpu()
    for p in range(P):
        k = int(expert.view(-1)[p])
        if k >= E:
            assert bool((act[p] == 7).all()) and bool((y[p] == 7).all())
            continue
        z = x[p // top].double().cpu() @ up[k].double().cpu().T
        want = z[:ff] * torch.sigmoid(z[:ff]) * z[ff:] if glu else torch.relu(z) ** 2
        assert float(((a64[p] - want).abs() / (want.abs() * 2.0 ** -8 + 1e-6 * D * (1 + want.abs().max().sqrt()))).max()) <= 1.0
        ref = a64[p] @ down[k].double().cpu().T
        assert float((y[p].double().cpu() - ref).abs().max()) <= 1e-6 * ff * float(a64.abs().max().clamp(min=1))
    for j in range(slices):
        z = x.double().cpu() @ s_up.double().cpu().T
        want = (z[:, :sff] * torch.sigmoid(z[:, :sff]) * z[:, sff:])[:, j * ff:(j + 1) * ff]
        got = a64[P + j * T:P + (j + 1) * T]
        assert float(((got - want).abs() / (want.abs() * 2.0 ** -8 + 1e-6 * D * (1 + want.abs().max().sqrt()))).max()) <= 1.0
        ref = got @ s_down[:, j * ff:(j + 1) * ff].double().cpu().T
        assert float((y[P + j * T:P + (j + 1) * T].double().cpu() - ref).abs().max()) <= 1e-6 * ff * float(a64.abs().max().clamp(min=1))
    if kind == "even" and T * top <= 64 and not slices:      # tables that cut no expert's pairs
        at, yt = both(False)
        assert torch.equal(act, at) and torch.equal(y, yt)
