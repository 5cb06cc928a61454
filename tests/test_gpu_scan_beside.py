"""Decode steps of a layer with a state-space scan beside its attention: the launches that do several things against the launches that do one each - the
same bits, states and caches included - and what is left to launches of their own."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def L():
    from pegainfer_amd import ffi
    return ffi.lib()


def ok(rc):
    assert rc == 0, rc


def step(n, heads, kv, hd, H, G, ns, vd, norm_heads, n_split, ff=70, taps=4, hv=None):
    """run(together) -> everything that the step leaves; the descriptions of the last run"""
    from pegainfer_amd import ops_blocks as B
    hv = hv or hd
    g = torch.Generator().manual_seed(n * hd + ns + vd)
    draw = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    inner, ch = H * vd, H * vd + 2 * G * ns
    offs, at = [], 0
    for w in (heads * hd, kv * hd, kv * hv, inner, ch, H, ff, ff):       # q k v z xBC dt gate up
        offs.append(at)
        at += -(-w // 8) * 8
    proj, cw, cb, A, dtb, Dk, nw, qn = draw(n, at), draw(ch, taps), draw(ch), draw(H), draw(H), draw(H), draw(inner), draw(hd)
    start = [int(t) for t in torch.randint(0, 400, (n,), generator=g)]
    rg = B.Ragged([1] * n, starts=start, slots=torch.randperm(n, generator=g).tolist())
    pages = [-(-(s + 1) // 16) for s in start]
    ind = torch.tensor([sum(pages[:i]) for i in range(n + 1)], dtype=torch.int32).cuda()
    ids = torch.randperm(sum(pages), generator=g).int().cuda()
    f = torch.tensor([100.0 ** (-i / 8) for i in range(8)]).cuda()
    tiles = B.attention_tiles(rg.lens, heads // kv, "cuda", 16)
    stride = 16 * kv * (hd + hv)
    cache0, mem0, tail0 = draw(sum(pages), stride), torch.randn(n, H * ns * vd, generator=g).cuda(), torch.randn(n, (taps - 1) * ch, generator=g).cuda()
    keep = {}

    def run(together):
        cache, mem, tail = cache0.clone(), mem0.clone(), tail0.clone()
        q32, x32, o = (torch.zeros(n, w, device="cuda") for w in (heads * hd, ch, inner))
        act, mix, out = (torch.zeros(n, w, dtype=torch.bfloat16, device="cuda") for w in (ff, heads * hv, inner))
        s, a = B._stream(), ctypes.addressof
        p = B.QkPrepDesc(proj=proj.data_ptr(), proj_dtype=0, proj_stride=at, q_off=offs[0], k_off=offs[1], v_off=offs[2], heads=heads, kv_heads=kv, dim=hd, vdim=hv,
                         q_norm=qn.data_ptr(), k_norm=qn.data_ptr(), eps=1e-5, inv_freq=f.data_ptr(), rot_dims=16, rot_layout=1, rot_amp=1.0,
                         positions=rg.positions.data_ptr(), row_entry=rg.row_entry.data_ptr(), page_indptr=ind.data_ptr(), page_ids=ids.data_ptr(),
                         cache=cache.data_ptr(), page_stride=stride, k_cache_off=0, v_cache_off=16 * kv * hd, page_size=16, q_out=q32.data_ptr(), n_rows=n, dtype=0)
        c = B.ConvGluStepDesc(in_=proj[:, offs[4]:].data_ptr(), in_row_stride=at, w=cw.data_ptr(), out_bias=cb.data_ptr(), state=tail.data_ptr(),
                              slot_stride=tail.stride(0), out=x32.data_ptr(), out_row_stride=ch, channels=ch, taps=taps, mode=2, entry_slot=rg.entry_slot.data_ptr(),
                              gate=proj[:, offs[6]:].data_ptr(), up=proj[:, offs[7]:].data_ptr(), glu_out=act.data_ptr(), glu_row_stride=ff, I=ff, act=1, n_entries=n,
                              dtype=0)
        d = B.SsdScanDesc(xbc=x32.data_ptr(), xbc_stride=ch, proj=proj.data_ptr(), proj_stride=at, dt_off=offs[5], A_log=A.data_ptr(), dt_bias=dtb.data_ptr(),
                          D=Dk.data_ptr(), state=mem.data_ptr(), slot_stride=mem.stride(0), o=o.data_ptr(), heads=H, groups=G, n_state=ns, vdim=vd,
                          entry_row0=rg.entry_row0.data_ptr(), entry_slot=rg.entry_slot.data_ptr(), n_entries=n, dtype=0)
        gate = proj[:, offs[3]:]
        b = B.ScanBesideDesc(scan=a(d), norm_w=nw.data_ptr(), gate=gate.data_ptr(), gate_stride=at, out=out.data_ptr(), out_stride=inner, factor=0.5, eps=1e-5,
                             w_per_head=1, gate_kind=0, gate_first=1, heads=norm_heads, vdim=inner // norm_heads, rows=n)
        ws = torch.zeros(L().pegainfer_paged_attention_workspace(tiles[0].numel(), kv, hv, 1, max(n_split, 2)), device="cuda")
        opt = B.AttnOptions(n_split=n_split, workspace=ws.data_ptr(), scan_beside=a(b) if together else None)
        keep.update(p=p, c=c, d=d, b=b, opt=opt)
        if together:
            assert L().pegainfer_qk_prep_conv_ok(a(p), a(c)) and L().pegainfer_paged_attention_scan_ok(a(opt), 0)
            ok(L().pegainfer_qk_prep_conv(a(p), a(c), s))
        else:
            ok(L().pegainfer_qk_prep(a(p), s))
            ok(L().pegainfer_conv_glu_step(a(c), s))
        ok(L().pegainfer_paged_attention_opt(q32.data_ptr(), cache.data_ptr(), stride, 0, 16 * kv * hd, 16, rg.positions.data_ptr(), rg.row_entry.data_ptr(),
                                             ind.data_ptr(), ids.data_ptr(), heads, kv, hd, hv, hd ** -0.5, 1.0, *(t.data_ptr() for t in tiles), tiles[0].numel(),
                                             mix.data_ptr(), heads * hv, a(opt), 0, s))
        if not together:
            ok(L().pegainfer_ssd_scan_form(a(d), s))
            ok(L().pegainfer_head_gate_rms(o.data_ptr(), nw.data_ptr(), 1, gate.data_ptr(), at, 0, 1, 0.5, 1e-5, out.data_ptr(), inner, norm_heads, inner // norm_heads, n,
                                           0, s))
        return cache, mem, tail, q32, x32, o, act, mix, out

    return run, keep


@pytest.mark.parametrize("args", [(1, 16, 4, 128, 32, 1, 128, 64, 4, 16), (3, 4, 2, 32, 3, 3, 33, 20, 1, 2), (2, 6, 6, 64, 4, 2, 64, 16, 4, 5), (5, 8, 1, 256, 2, 1, 100, 48, 2, 64)])
def test_both_as_by_themselves(args):
    run, _ = step(*args)
    for a, b in zip(run(False), run(True)):
        assert torch.equal(a, b) and torch.isfinite(a.float()).all() and float(a.float().abs().max()) > 0


@pytest.mark.parametrize("hd,hv", [(192, 128), (180, 100), (80, 200), (66, 256), (256, 256)])
def test_tiles_near_64_KB_beside_the_largest_scan(hd, hv):
    """the keys' and values' tiles take 48 KB and less or more, the scan's 17.5 KB come to them"""
    run, _ = step(2, 4, 2, hd, 4, 2, 128, 16, 2, 4, hv=hv)
    for a, b in zip(run(False), run(True)):
        assert torch.equal(a, b) and torch.isfinite(a.float()).all()


def test_what_is_left_to_launches_of_their_own():
    run, keep = step(2, 4, 2, 64, 4, 2, 64, 16, 2, 4)
    run(False)
    keep["opt"].scan_beside = ctypes.addressof(keep["b"])
    scan = lambda dtype=0: L().pegainfer_paged_attention_scan_ok(ctypes.addressof(keep["opt"]), dtype)
    conv = lambda: L().pegainfer_qk_prep_conv_ok(ctypes.addressof(keep["p"]), ctypes.addressof(keep["c"]))
    assert scan() and not scan(1) and conv()
    for d, field, value, yes in (("opt", "n_split", 1, scan), ("opt", "maps", 2, scan), ("opt", "plain", 1, scan), ("opt", "tile_rows", 64, scan), ("d", "n_state", 32, scan),
                                 ("d", "n_state", 129, scan), ("d", "n_long", 1, scan), ("d", "dtype", 1, scan), ("b", "vdim", 513, scan), ("p", "proj_dtype", 1, conv),
                                 ("p", "proj_stride", 63, conv), ("c", "dtype", 1, conv), ("c", "I", 0, conv)):
        old = getattr(keep[d], field)
        setattr(keep[d], field, value)
        assert not yes(), (d, field)
        setattr(keep[d], field, old)
