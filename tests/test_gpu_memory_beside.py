"""Decode steps of a layer with an attention beside a matrix memory, and of the ends of the layer stack: the launches that do several things against the
launches that do one each - the same bits, state included."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def L():
    from pegainfer_amd import ffi
    return ffi.lib()


def ok(rc):
    assert rc == 0, rc


@pytest.mark.parametrize("n,H,dim,vdim,heads,kv,hd", [(1, 8, 128, 256, 16, 4, 256), (3, 3, 100, 20, 4, 2, 64), (2, 1, 16, 12, 2, 1, 32), (5, 2, 256, 512, 6, 3, 128),
                                                      (1, 5, 33, 70, 3, 3, 40)])
def test_scan_beside_the_preparation_and_what_is_left_of_both(n, H, dim, vdim, heads, kv, hd):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(n * dim + vdim)
    draw = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    offs, at = [], 0
    for w in (H * dim, H * dim, H * vdim, H, H, H * vdim, heads * hd, kv * hd, kv * hd):     # q k v i f gate | q k v of the attention
        offs.append(at)
        at += -(-w // 4) * 4
    proj, i_b, f_b, rnorm, qn, kn = draw(n, at), draw(H), draw(H), draw(H * vdim), draw(hd), draw(hd)
    start = [int(t) for t in torch.randint(0, 40, (n,), generator=g)]
    rg = B.Ragged([1] * n, starts=start, slots=torch.randperm(n, generator=g).tolist())
    pages = [-(-(s + 1) // 16) for s in start]
    ind = torch.tensor([sum(pages[:i]) for i in range(n + 1)], dtype=torch.int32).cuda()
    ids = torch.randperm(sum(pages), generator=g).int().cuda()
    f = torch.tensor([100.0 ** (-i / 8) for i in range(8)]).cuda()
    state0 = torch.randn(n, H * (dim * vdim + dim + 1), generator=g).cuda()
    rows = draw(n, heads * hd)

    def run(together):
        state, o = state0.clone(), torch.zeros(n, H * vdim, device="cuda")
        cache = torch.zeros(sum(pages), 2 * 16 * kv * hd, dtype=torch.bfloat16, device="cuda")
        q16, mix = torch.zeros(n, heads * hd, dtype=torch.bfloat16, device="cuda"), torch.zeros(n, heads * hd + H * vdim, dtype=torch.bfloat16, device="cuda")
        m = B.MatrixMemoryDesc(proj=proj.data_ptr(), proj_stride=at, q_off=offs[0], k_off=offs[1], v_off=offs[2], i_off=offs[3], f_off=offs[4],
                               i_bias=i_b.data_ptr(), f_bias=f_b.data_ptr(), cap=8.0, state=state.data_ptr(), slot_stride=state.stride(0), o=o.data_ptr(),
                               heads=H, dim=dim, vdim=vdim, entry_row0=rg.entry_row0.data_ptr(), entry_slot=rg.entry_slot.data_ptr(), n_entries=n, dtype=0)
        p = B.QkPrepDesc(proj=proj.data_ptr(), proj_dtype=0, proj_stride=at, q_off=offs[6], k_off=offs[7], v_off=offs[8], heads=heads, kv_heads=kv, dim=hd, vdim=hd,
                         q_norm=qn.data_ptr(), k_norm=kn.data_ptr(), eps=1e-5, inv_freq=f.data_ptr(), rot_dims=16, rot_layout=0, rot_amp=1.0,
                         positions=rg.positions.data_ptr(), row_entry=rg.row_entry.data_ptr(), page_indptr=ind.data_ptr(), page_ids=ids.data_ptr(),
                         cache=cache.data_ptr(), page_stride=cache.stride(0), k_cache_off=0, v_cache_off=16 * kv * hd, page_size=16, q_out_stored=q16.data_ptr(),
                         n_rows=n, dtype=0)
        s, a = B._stream(), ctypes.addressof
        gate, right = proj[:, offs[5]:], mix[:, heads * hd:]
        if together:
            assert L().pegainfer_gated_matrix_memory_beside_ok(a(m), a(p))
            ok(L().pegainfer_gated_matrix_memory_beside(a(m), a(p), s))
            fin = B.MemoryFinishDesc(norm_w=rnorm.data_ptr(), gate=gate.data_ptr(), gate_stride=at, gate_kind=1, factor=0.5, eps=1e-5, out=right.data_ptr(),
                                     out_stride=mix.stride(0), rows=rows.data_ptr(), rows_stride=heads * hd, scaled=mix.data_ptr(), scaled_stride=mix.stride(0),
                                     scale_cols=heads * hd, scale=0.75)
            ok(L().pegainfer_gated_matrix_memory_finish(a(m), a(fin), s))
        else:
            ok(L().pegainfer_qk_prep(a(p), s))
            ok(L().pegainfer_gated_matrix_memory_form(a(m), s))
            ok(L().pegainfer_scale_rows(rows.data_ptr(), heads * hd, mix.data_ptr(), mix.stride(0), heads * hd, n, 0.75, 0, s))
            ok(L().pegainfer_head_rms_gate(o.data_ptr(), rnorm.data_ptr(), 1, gate.data_ptr(), at, 1, 0.5, 1e-5, right.data_ptr(), mix.stride(0), H, vdim, n, 0, s))
        return state, cache, q16, mix

    for x, y in zip(run(False), run(True)):
        assert torch.equal(x, y) and torch.isfinite(x.float()).all()


def test_what_is_left_to_launches_of_their_own():
    from pegainfer_amd import ops_blocks as B
    m = B.MatrixMemoryDesc(cap=1.0, heads=2, dim=16, vdim=32, n_entries=1, dtype=0)
    p = B.QkPrepDesc(heads=2, kv_heads=1, dim=32, vdim=32, page_size=16, n_rows=1, proj_stride=64, page_stride=64)
    yes = lambda: L().pegainfer_gated_matrix_memory_beside_ok(ctypes.addressof(m), ctypes.addressof(p))
    assert yes()
    for d, field, value in ((m, "dtype", 1), (m, "vdim", 516), (m, "n_long", 1), (m, "dim", 260), (p, "dtype", 1), (p, "proj_dtype", 1), (p, "dim", 31), (p, "proj_stride", 63)):
        old = getattr(d, field)
        setattr(d, field, value)
        assert not yes(), field
        setattr(d, field, old)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,d,taps,groups", [(1, 2560, 4, 4), (3, 70, 1, 7), (5, 300, 9, 3)])
def test_first_convolution_and_last_norm(dtype, n, d, taps, groups):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(d)
    draw = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    embed, w, gain, td, s = draw(50, d), draw(d, taps), draw(d), B._dt(draw(1)), B._stream()
    tok = torch.randint(0, 50, (n,), generator=g).int().cuda()
    slots = torch.randperm(n, generator=g).int().cuda()
    tail0 = torch.randn(n, max(taps - 1, 1) * d, generator=g).cuda()
    res = []
    for together in (False, True):
        tail, x, hb = tail0.clone(), torch.zeros(n, d, device="cuda"), torch.zeros(n, d, dtype=dtype, device="cuda")
        if together:
            ok(L().pegainfer_embed_conv_step(embed.data_ptr(), tok.data_ptr(), x.data_ptr(), w.data_ptr(), tail.data_ptr(), tail.stride(0), hb.data_ptr(), d, taps, 1,
                                             slots.data_ptr(), n, td, s))
        else:
            ok(L().pegainfer_embed_f32(embed.data_ptr(), tok.data_ptr(), x.data_ptr(), d, n, td, s))
            ok(L().pegainfer_time_conv_step(x.data_ptr(), 1, d, w.data_ptr(), td, tail.data_ptr(), tail.stride(0), hb.data_ptr(), td, d, d, taps, 1, slots.data_ptr(), n, s))
        res.append((tail, x, hb))
    for a, b in zip(*res):
        assert torch.equal(a, b)
    x, idx = torch.randn(n, d, generator=g).cuda(), torch.randint(0, n, (4,), generator=g).int().cuda()
    xw, a, b = torch.empty(4, d, device="cuda"), torch.zeros(4, d, dtype=dtype, device="cuda"), torch.zeros(4, d, dtype=dtype, device="cuda")
    ok(L().pegainfer_gather_rows_f32(x.data_ptr(), idx.data_ptr(), xw.data_ptr(), d, 4, s))
    ok(L().pegainfer_group_rms_add(None, xw.data_ptr(), 1, gain.data_ptr(), groups, 1e-5, None, a.data_ptr(), d, 4, td, None, 0, None, 0, None, None, s))
    ok(L().pegainfer_group_rms_rows(x.data_ptr(), idx.data_ptr(), gain.data_ptr(), groups, 1e-5, b.data_ptr(), d, 4, td, s))
    assert torch.equal(a, b) and float(a.float().abs().max()) > 0
