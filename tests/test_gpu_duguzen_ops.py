"""Each Duguzen mechanism alone on the GPU against the plain restatement (oracle/duguzen_ref.py) or a direct torch fp32 /
fp64 formula: Dynamic-Tanh norms, the strided / batched / grouped GEMM, latent prep (RMS norm + rotation + cache write), the
latent attention (pages, key splits, crafted far keys), the grouped sigmoid router, expert sorting and combine."""
import math

import numpy as np
import pytest
import torch

import duguzen_common as C
from oracle import duguzen_ref as R

pytestmark = pytest.mark.gpu

DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def dev(t, dtype=None):
    t = torch.as_tensor(t)
    return (t.to(dtype) if dtype else t).cuda().contiguous()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_dyt_norm_and_fused_boundary(dtype):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(0)
    rows, d = 37, 52
    x = torch.randn(rows, d, generator=g) * 3
    y = C.bf16_round(torch.randn(rows, d, generator=g) * 2)
    P = [C.bf16_round(v) for v in (torch.tensor(0.7), 1 + 0.2 * torch.randn(d, generator=g), 0.1 * torch.randn(d, generator=g))]
    N = [C.bf16_round(v) for v in (torch.tensor(0.4), 1 + 0.2 * torch.randn(d, generator=g), 0.1 * torch.randn(d, generator=g))]
    td = DT[dtype]
    ref1 = torch.tanh(P[0].double() * x.double()) * P[1].double() + P[2].double()
    got1 = B.dyt_norm(dev(x), *[dev(v, td) for v in P]).float().cpu()
    tol = 1e-6 if dtype == "float32" else 1e-2
    assert (got1.double() - ref1).abs().max() < tol
    xs = dev(x)
    got2 = B.dyt_add_norm(xs, dev(y, td), [dev(v, td) for v in P], [dev(v, td) for v in N]).float().cpu()
    x2 = x.double() + torch.tanh(P[0].double() * y.double()) * P[1].double() + P[2].double()
    assert (xs.cpu().double() - x2).abs().max() < 2e-6            # the residual sum is fp32 in both instances
    ref2 = torch.tanh(N[0].double() * x2) * N[1].double() + N[2].double()
    assert (got2.double() - ref2).abs().max() < tol
    xs2 = dev(x)
    assert B.dyt_add_norm(xs2, dev(y, td), [dev(v, td) for v in P]) is None
    assert torch.equal(xs2, xs)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_strided_gemm_dense_batched_transposed(dtype):
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(1)
    td = DT[dtype]
    for (T, M, K) in [(1, 5, 3), (70, 66, 50), (64, 64, 16), (130, 7, 129)]:
        x, w = C.bf16_round(torch.randn(T, K, generator=g)), C.bf16_round(torch.randn(M, K, generator=g))
        got = B.linear(dev(x, td), dev(w, td), out_dtype=torch.float32).cpu()
        assert (got.double() - x.double() @ w.double().T).abs().max() < 1e-4 * K
        sq = B.linear(dev(x, td), dev(w, td), out_dtype=torch.float32, epilogue=B.EPI_RELU_SQ).cpu()
        assert (sq.double() - torch.relu(x.double() @ w.double().T) ** 2).abs().max() < 1e-3 * K
    # per-head product over slices of a wider row with the weight read transposed, then one with a sigmoid gate
    T, H, dn, dr, r = 9, 3, 10, 6, 14
    row = C.bf16_round(torch.randn(T, H * (dn + dr) + 5, generator=g))
    uk = C.bf16_round(torch.randn(H * dn, r, generator=g))
    qc = torch.zeros(T, H, r + dr, device="cuda")
    xd, wd = dev(row, td), dev(uk, td)
    d = B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=qc.data_ptr(), x_dtype=B._dt(xd), w_dtype=B._dt(wd), y_dtype=1, m=r,
                   k=dn, rows=T, groups=H, x_row_stride=row.shape[1], x_group_stride=dn + dr, w_m_stride=1, w_k_stride=r,
                   w_group_stride=dn * r, y_row_stride=H * (r + dr), y_group_stride=r + dr)
    B.gemm_strided(d)
    q = row[:, :H * (dn + dr)].reshape(T, H, dn + dr)[..., :dn].double()
    ref = torch.einsum("thd,hdr->thr", q, uk.double().reshape(H, dn, r))
    assert (qc.cpu()[..., :r].double() - ref).abs().max() < 1e-4 and float(qc[..., r:].abs().max()) == 0.0
    gate = C.bf16_round(torch.randn(T, H + 2, generator=g))
    ol, uv = torch.randn(T, H, r, generator=g), C.bf16_round(torch.randn(H * 7, r, generator=g))
    out = torch.zeros(T, H * 7, device="cuda", dtype=td)
    old, uvd, gd = dev(ol), dev(uv, td), dev(gate, td)
    d = B.GemmDesc(x=old.data_ptr(), w=uvd.data_ptr(), y=out.data_ptr(), x_dtype=1, w_dtype=B._dt(uvd), y_dtype=B._dt(out), m=7,
                   k=r, rows=T, groups=H, x_row_stride=H * r, x_group_stride=r, w_m_stride=r, w_k_stride=1, w_group_stride=7 * r,
                   y_row_stride=H * 7, y_group_stride=7, epilogue=B.EPI_SIGMOID_GATE, gate=gd.data_ptr() + 2 * gd.element_size(),
                   gate_dtype=B._dt(gd), gate_row_stride=H + 2)
    B.gemm_strided(d)
    ref = torch.einsum("thr,hvr->thv", ol.double(), uv.double().reshape(H, 7, r)) * torch.sigmoid(gate[:, 2:].double())[..., None]
    assert (out.float().cpu().double().reshape(T, H, 7) - ref).abs().max() < (1e-4 if dtype == "float32" else 0.05)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_router_matches_the_plain_rule(dtype):
    from pegainfer_amd import ops_blocks as B
    td = DT[dtype]
    g = torch.Generator().manual_seed(2)
    cases = [(12, 4, 3, 4), (16, 4, 3, 4), (6, 3, 2, 2), (5, 1, 1, 1), (4, 4, 4, 3), (8, 8, 3, 2), (9, 3, 1, 3)]
    for (E, G, keep, top) in cases:
        d = 40
        h = C.bf16_round(torch.randn(33, d, generator=g))
        w = {"r.router": C.bf16_round(torch.randn(E, d, generator=g) * 0.5),
             "r.correction": C.bf16_round(torch.randn(E, generator=g) - 0.8)}
        rt = {"experts": E, "top": top, "groups": {"count": G, "keep": keep}}
        idx, wt = R.route(h.double(), w, "r", rt)
        e, ww = B.route(dev(h, td), dev(w["r.router"], td), dev(w["r.correction"], td), G, keep, top)
        assert torch.equal(e.cpu().long(), idx), (E, G, keep, top)
        assert (ww.cpu().double() - wt).abs().max() < 1e-5
        e2, _ = B.route(dev(h, td), dev(w["r.router"], td), None, G, keep, top)      # no correction: choose by the scores
        idx2, _ = R.route(h.double(), {"r.router": w["r.router"]}, "r", rt)
        assert torch.equal(e2.cpu().long(), idx2)


def test_expert_sort_grouped_gemm_and_combine():
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(3)
    rows, top, E, d, ff = 150, 3, 5, 24, 10          # expert 4 gets > 64 pairs (two tiles), expert 3 none
    expert = torch.randint(0, 3, (rows, top), generator=g, dtype=torch.int32)
    expert[:, 2] = 4
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), E)
    n = int(nt.item())
    pp, tgc, t0c, trc = pos_pair.cpu(), tg.cpu()[:n], t0.cpu()[:n], tr.cpu()[:n]
    assert sorted(pp.tolist()) == list(range(rows * top)) and torch.equal(pos_row.cpu(), pp // top)
    assert int(trc.sum()) == rows * top and int(trc.max()) <= 64 and 3 not in tgc.tolist()
    for i in range(n):
        assert all(int(expert.reshape(-1)[pp[p]]) == int(tgc[i]) for p in range(int(t0c[i]), int(t0c[i] + trc[i])))
    x = C.bf16_round(torch.randn(rows, d, generator=g))
    w = C.bf16_round(torch.randn(E, ff, d, generator=g))
    y = torch.zeros(rows * top, ff, device="cuda")
    xd, wd = dev(x, torch.bfloat16), dev(w, torch.bfloat16)
    dsc = B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=1, m=ff, k=d,
                     x_row_stride=d, w_m_stride=d, w_k_stride=1, w_group_stride=ff * d, y_row_stride=ff,
                     tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(),
                     max_tiles=max_tiles, x_row_index=pos_row.data_ptr(), y_row_index=pos_pair.data_ptr())
    B.gemm_strided(dsc)
    ref = torch.einsum("pd,pfd->pf", x.double().repeat_interleave(top, 0), w.double()[expert.reshape(-1).long()])
    assert (y.cpu().double() - ref).abs().max() < 1e-4
    wt = torch.rand(rows, top, generator=g)
    out = B.route_combine(y, wt.cuda(), torch.float32).cpu()
    assert (out.double() - (ref.reshape(rows, top, ff) * wt.double()[..., None]).sum(1)).abs().max() < 1e-4


def _paged(entries, page_size, dtype, perm_seed=0):
    """entries [n, E] -> (cache tensor, page ids) with the pages in a scrambled order inside a larger pool"""
    n, E = entries.shape
    npages = (n + page_size - 1) // page_size
    pool = npages + 3
    order = np.random.default_rng(perm_seed).permutation(pool)[:npages]
    cache = torch.zeros(pool, page_size, E)
    for j in range(n):
        cache[order[j // page_size], j % page_size] = entries[j]
    return dev(cache, dtype), torch.tensor(order, dtype=torch.int32).cuda()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_latent_prep_norm_rotation_and_cache_write(dtype):
    from pegainfer_amd import ops_blocks as B
    td = DT[dtype]
    g = torch.Generator().manual_seed(4)
    H, dn, dr, r, rd, ps, base, eps = 3, 10, 12, 20, 8, 16, 777.0, 1e-5
    T, start = 21, 27                                   # positions 27 .. 47: the portion starts inside a page
    proj = C.bf16_round(torch.randn(T, H * (dn + dr) + r + dr + H, generator=g))
    cw = C.bf16_round(1 + 0.2 * torch.randn(r, generator=g))
    pos = torch.arange(start, start + T)
    E = r + dr
    cache, pages = _paged(torch.zeros(start + T, E), ps, td)
    inv = torch.tensor([base ** (-2.0 * i / rd) for i in range(rd // 2)], dtype=torch.float32).cuda()
    qc = torch.zeros(T, H, E, device="cuda")
    B.latent_prep(dev(proj, td), H * (dn + dr), dev(cw, td), eps, inv, rd, pos.int().cuda(), torch.zeros(T, dtype=torch.int32).cuda(),
                  torch.tensor([0, len(pages)], dtype=torch.int32).cuda(), pages, cache, ps * E, 0, ps, qc, H, dn, dr, r)
    dkv = proj[:, H * (dn + dr):H * (dn + dr) + E].double()
    c_ref = R.rms(dkv[:, :r], cw.double(), eps)
    kr_ref = R.rope_half(dkv[:, r:], pos, base, rd)
    q_ref = R.rope_half(proj[:, :H * (dn + dr)].double().reshape(T, H, dn + dr)[..., dn:], pos, base, rd)
    flat = cache.float().cpu()
    got = torch.stack([flat[int(pages[p // ps]), p % ps] for p in range(start, start + T)]).double()
    tol = 2e-5 if dtype == "float32" else 2e-2
    assert (got[:, :r] - c_ref).abs().max() < tol and (got[:, r:] - kr_ref).abs().max() < tol
    assert (qc.cpu()[..., r:].double() - q_ref).abs().max() < 2e-5          # the query side stays fp32
    untouched = torch.stack([flat[int(pages[p // ps]), p % ps] for p in range(start)])
    assert float(untouched.abs().max()) == 0.0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n_keys", [1, 17, 256, 257, 1024, 1025, 1300])
def test_latent_attention_matches_softmax(dtype, n_keys):
    from pegainfer_amd import ops_blocks as B
    td = DT[dtype]
    g = torch.Generator().manual_seed(n_keys)
    H, r, dr, ps = 3, 24, 8, 16
    E = r + dr
    entries = C.bf16_round(torch.randn(n_keys, E, generator=g))
    cache, pages = _paged(entries, ps, td, perm_seed=n_keys)
    rows = sorted({0, n_keys // 2, n_keys - 1})
    qc = torch.randn(len(rows), H, E, generator=g)
    o = B.latent_attention(dev(qc), cache, ps * E, 0, ps, torch.tensor(rows, dtype=torch.int32).cuda(),
                           torch.zeros(len(rows), dtype=torch.int32).cuda(), torch.tensor([0, len(pages)], dtype=torch.int32).cuda(),
                           pages, r, dr, 0.3, n_keys).cpu()
    for i, p in enumerate(rows):
        s = torch.einsum("he,je->hj", qc[i].double(), entries[:p + 1].double()) * 0.3
        ref = torch.softmax(s, -1) @ entries[:p + 1, :r].double()
        assert (o[i].double() - ref).abs().max() < 2e-5, (n_keys, p)


@pytest.mark.parametrize("far", [0, 15, 16, 255, 256, 1023, 1024, 1100])
def test_one_far_key_stands_out(far):
    """one key is made to dominate the softmax: the output must be that key's latent, wherever it sits - the first token,
    either side of a page border, of a round of keys and of a key split - and must ignore it when it is not yet visible"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(far)
    n, H, r, dr, ps = 1200, 2, 16, 8, 16
    E = r + dr
    entries = C.bf16_round(torch.randn(n, E, generator=g) * 0.2)
    probe = torch.zeros(E)
    probe[3], probe[r + 1] = 8.0, 8.0
    entries[far] = probe
    cache, pages = _paged(entries, ps, torch.float32, perm_seed=far)
    qc = torch.zeros(3, H, E)
    qc[:, :, 3] = qc[:, :, r + 1] = 4.0
    rows = [n - 1, far, max(far - 1, 0)]                # sees it from afar, sees it as its own position, does not see it
    o = B.latent_attention(dev(qc), cache, ps * E, 0, ps, torch.tensor(rows, dtype=torch.int32).cuda(),
                           torch.zeros(3, dtype=torch.int32).cuda(), torch.tensor([0, len(pages)], dtype=torch.int32).cuda(),
                           pages, r, dr, 1.0, n).cpu()
    assert (o[0] - probe[:r]).abs().max() < 1e-3 and (o[1] - probe[:r]).abs().max() < 1e-3
    if far > 0:
        assert float(o[2][:, 3].abs().max()) < 1.0


def test_latent_attention_rows_of_several_requests():
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(9)
    H, r, dr, ps = 2, 8, 4, 16
    E = r + dr
    lens = [40, 3, 17]
    ent = [C.bf16_round(torch.randn(n, E, generator=g)) for n in lens]
    pool = torch.zeros(12, ps, E)
    page_lists, nxt = [], 11
    for e in ent:                                        # pages handed out from the top, interleaved between requests
        pl = []
        for j in range(0, len(e), ps):
            pool[nxt, :len(e[j:j + ps])] = e[j:j + ps]
            pl.append(nxt)
            nxt -= 1
        page_lists.append(pl)
    indptr = np.cumsum([0] + [len(p) for p in page_lists]).astype(np.int32)
    rows = [(0, 39), (1, 0), (2, 16), (0, 15), (1, 2), (2, 15), (0, 16)]
    qc = torch.randn(len(rows), H, E, generator=g)
    o = B.latent_attention(dev(qc), dev(pool, torch.bfloat16), ps * E, 0, ps, torch.tensor([p for _, p in rows], dtype=torch.int32).cuda(),
                           torch.tensor([q for q, _ in rows], dtype=torch.int32).cuda(), torch.tensor(indptr).cuda(),
                           torch.tensor(sum(page_lists, []), dtype=torch.int32).cuda(), r, dr, 0.5, 40).cpu()
    for i, (q, p) in enumerate(rows):
        s = torch.einsum("he,je->hj", qc[i].double(), ent[q][:p + 1].double()) * 0.5
        assert (o[i].double() - torch.softmax(s, -1) @ ent[q][:p + 1, :r].double()).abs().max() < 2e-5


@pytest.mark.parametrize("split_keys", [0, 128])
@pytest.mark.parametrize("shape", [(3, 32, 8, [70, 1, 9]), (8, 64, 32, [300, 2]), (5, 16, 16, [13, 13, 1, 1]), (16, 128, 64, [5, 40])])
def test_latent_attention_matrix_core_form(shape, split_keys):
    """the tiled bf16 form against the direct softmax: several requests in one launch, portions that start deep inside a
    context, tiles that end inside an entry, key splits; q and the weights are rounded to bf16 inside, hence the tolerance"""
    from pegainfer_amd import ops_blocks as B
    H, r, dr, lens = shape
    g = torch.Generator().manual_seed(H * 100 + r)
    E, ps = r + dr, 16
    starts = [0 if i % 2 == 0 else 137 for i in range(len(lens))]          # odd entries continue a context of 137 tokens
    ctx = [s + n for s, n in zip(starts, lens)]
    ent = [C.bf16_round(torch.randn(n, E, generator=g) * 0.7) for n in ctx]
    npages = [(n + ps - 1) // ps for n in ctx]
    pool = torch.zeros(sum(npages) + 2, ps, E)
    order = np.random.default_rng(H).permutation(sum(npages) + 2)
    page_lists, at = [], 0
    for e, k in zip(ent, npages):
        pl = [int(x) for x in order[at:at + k]]
        at += k
        for j in range(len(e)):
            pool[pl[j // ps], j % ps] = e[j]
        page_lists.append(pl)
    indptr = np.cumsum([0] + npages).astype(np.int32)
    pos = [s + k for s, n in zip(starts, lens) for k in range(n)]
    req = [i for i, n in enumerate(lens) for _ in range(n)]
    T = len(pos)
    qc = torch.randn(T, H, E, generator=g)
    assert ffi_ok(B, r, dr, ps * E)
    args = (dev(pool, torch.bfloat16), ps * E, 0, ps, torch.tensor(pos, dtype=torch.int32).cuda(), torch.tensor(req, dtype=torch.int32).cuda(),
            torch.tensor(indptr).cuda(), torch.tensor(sum(page_lists, []), dtype=torch.int32).cuda(), r, dr, 0.25, max(ctx))
    o = B.latent_attention(dev(qc), *args, split_keys=split_keys, tiles=B.row_tiles(lens, H)).cpu()
    plain = B.latent_attention(dev(qc), *args, split_keys=split_keys).cpu()
    for i in range(T):
        e = ent[req[i]][:pos[i] + 1].double()
        ref = torch.softmax(torch.einsum("he,je->hj", qc[i].double(), e) * 0.25, -1) @ e[:, :r]
        assert (plain[i].double() - ref).abs().max() < 2e-5, i
        assert (o[i].double() - ref).abs().max() < 2.5e-2, (i, pos[i], float((o[i].double() - ref).abs().max()))
    assert float((o - plain).abs().mean()) < 2e-3


# entries of 417 to 608 values take a second set of waves: both ends and one beyond each, ranks that fill their blocks and one that does not, tiles of keys
# that end in either half
@pytest.mark.parametrize("split_keys", [0, 128, 72])
@pytest.mark.parametrize("shape", [(16, 384, 32, [40, 5]), (8, 400, 24, [70, 1, 9]), (16, 512, 64, [33, 2, 64]), (4, 512, 96, [100, 33]), (4, 512, 104, [21])])
def test_latent_attention_two_sets_of_waves(shape, split_keys):
    test_latent_attention_matrix_core_form(shape, split_keys)


@pytest.mark.parametrize("split_keys", [0, 32, -3])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", [(8, 256, 64, [1, 1, 1]), (16, 512, 64, [1, 1]), (3, 16, 8, [5, 1, 9]), (40, 512, 128, [1]), (5, 272, 24, [3, 13, 1]),
                                   (24, 64, 0, [1, 1]), (64, 128, 64, [3])])
def test_latent_attention_few_rows_form(shape, dtype, split_keys):
    """tiles of a few rows (and any tile of an fp32 cache): one to four blocks of sixteen rows, entries that end inside a block, portions
    deep inside a context; split_keys < 0: the keys dealt to that many workgroups.  In fp32 the sums of at most 640 products of about
    one each and of 300 weights stay within 2e-5; q and the weights are rounded to bf16 in the other instance."""
    from pegainfer_amd import ops_blocks as B
    H, r, dr, lens = shape
    g = torch.Generator().manual_seed(H * 10 + r)
    E, ps = r + dr, 16
    starts = [0, 290, 33][:len(lens)]
    ctx = [s + n for s, n in zip(starts, lens)]
    ent = [C.bf16_round(torch.randn(n, E, generator=g) * 0.7) for n in ctx]
    npages = [(n + ps - 1) // ps for n in ctx]
    pool = torch.full((sum(npages), ps, E), float("nan"))                  # slots past an entry's context are never used
    order = np.random.default_rng(H).permutation(sum(npages))
    page_lists, at = [], 0
    for e, k in zip(ent, npages):
        page_lists.append([int(x) for x in order[at:at + k]])
        at += k
        for j in range(len(e)):
            pool[page_lists[-1][j // ps], j % ps] = e[j]
    pos = [s + k for s, n in zip(starts, lens) for k in range(n)]
    req = [i for i, n in enumerate(lens) for _ in range(n)]
    qc = torch.randn(len(pos), H, E, generator=g) / E ** 0.5
    indptr = torch.tensor(np.cumsum([0] + npages).astype(np.int32)).cuda()
    ids = torch.tensor(sum(page_lists, []), dtype=torch.int32).cuda()
    cache, tiles = dev(pool, DT[dtype]), B.row_tiles(lens, H)
    if split_keys < 0:
        o = B.latent_attention_dealt(dev(qc), cache, ps * E, 0, ps, B.Ragged(lens, starts=starts), indptr, ids, r, dr, 2.0, n_split=-split_keys, tiles=tiles)
    else:
        o = B.latent_attention(dev(qc), cache, ps * E, 0, ps, torch.tensor(pos, dtype=torch.int32).cuda(),
                               torch.tensor(req, dtype=torch.int32).cuda(), indptr, ids, r, dr, 2.0, max(ctx), split_keys=split_keys, tiles=tiles)
    tol = 2e-5 if dtype == "float32" else 2.5e-2
    for i in range(len(pos)):
        e = ent[req[i]][:pos[i] + 1].double()
        ref = torch.softmax(torch.einsum("he,je->hj", qc[i].double(), e) * 2.0, -1) @ e[:, :r]
        assert (o[i].cpu().double() - ref).abs().max() < tol, (i, pos[i], float((o[i].cpu().double() - ref).abs().max()))


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("H,r,dr", [(8, 256, 64), (3, 16, 8), (40, 512, 64)])
def test_fp32_latent_attention_keeps_later_entries_from_earlier_rows(H, r, dr, bad):
    """an entry that is infinite or no number, in the latent or in the rotated part, at the start, in the middle and at the end of a key tile: the rows
    before it are what they are without it, the rows from it on are no numbers"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(r)
    E, ps, T = r + dr, 16, 75
    ent, qc = torch.randn(T, E, generator=g) * 0.5, torch.randn(T, H, E, generator=g) / E ** 0.5
    npages = (T + ps - 1) // ps
    pos, req = torch.arange(T, dtype=torch.int32).cuda(), torch.zeros(T, dtype=torch.int32).cuda()
    indptr, ids = torch.tensor([0, npages], dtype=torch.int32).cuda(), torch.arange(npages, dtype=torch.int32).cuda()

    def run(e, **kw):
        pool = torch.zeros(npages * ps, E)
        pool[:T] = e
        return B.latent_attention(qc.cuda(), pool.cuda(), ps * E, 0, ps, pos, req, indptr, ids, r, dr, 1.0, T, tiles=B.row_tiles([T], H), **kw).cpu()

    for at, col in ((31, 3), (32, r - 1), (50, 0), (74, r + dr - 1)):
        e = ent.clone()
        e[at, col] = bad
        for kw in ({}, {"split_keys": 32}):
            sound, got = run(ent, **kw), run(e, **kw)
            assert float((got[:at] - sound[:at]).abs().max()) < 1e-5, (at, col)     # sums of 32 products in another order
            if col < r:
                assert not torch.isfinite(got[at:, :, col]).any()


def ffi_ok(B, r, dr, page_stride):
    from pegainfer_amd import ffi
    return ffi.lib().pegainfer_latent_attention_tiled_ok(r, dr, page_stride, 0, 0) == 1


def test_matrix_core_form_sees_a_far_key_and_masks_an_unseen_one():
    from pegainfer_amd import ops_blocks as B
    for far in (0, 31, 32, 127, 128, 700):
        g = torch.Generator().manual_seed(far)
        n, H, r, dr, ps = 800, 8, 16, 16, 16
        E = r + dr
        entries = C.bf16_round(torch.randn(n, E, generator=g) * 0.2)
        probe = torch.zeros(E)
        probe[3], probe[r + 1] = 8.0, 8.0
        entries[far] = probe
        cache, pages = _paged(entries, ps, torch.bfloat16, perm_seed=far)
        lo = max(far - 1, 0)
        T = n - lo                                       # one portion: positions lo .. n-1
        qc = torch.zeros(T, H, E)
        qc[:, :, 3] = qc[:, :, r + 1] = 4.0
        o = B.latent_attention(dev(qc), cache, ps * E, 0, ps, torch.arange(lo, n, dtype=torch.int32).cuda(),
                               torch.zeros(T, dtype=torch.int32).cuda(), torch.tensor([0, len(pages)], dtype=torch.int32).cuda(),
                               pages, r, dr, 1.0, n, split_keys=128, tiles=B.row_tiles([T], H)).cpu()
        seen = o[far - lo:]
        assert (seen - probe[:r]).abs().max() < 2e-2, far
        if far > 0:
            assert float(o[0][:, 3].abs().max()) < 1.0


@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 16])
@pytest.mark.parametrize("M,K", [(1, 8), (15, 40), (129, 520), (40, 2056), (33, 4104), (8200, 72)])
def test_few_rows_of_fp32_weights(T, M, K):
    """FMA with one, two and four rows and the fp32 matrix cores, a K that ends inside a piece, a chunk and beyond two of them (what lies behind it in
    the wider rows is no number), gathered and scattered rows, also from an expert table: sums of K products of about one in fp32"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(T * 1000 + M + K)
    x, w = torch.full((T + 2, K + 8), float("nan")), torch.full((3, M, K + 8), float("nan"))
    x[:, :K], w[..., :K] = torch.randn(T + 2, K, generator=g), torch.randn(3, M, K, generator=g)
    xd, wd = x.cuda(), w.cuda()
    base = dict(x=xd.data_ptr(), w=wd.data_ptr(), x_dtype=1, w_dtype=1, y_dtype=1, m=M, k=K, x_row_stride=K + 8, w_m_stride=K + 8, w_k_stride=1,
                w_group_stride=M * (K + 8), epilogue=B.EPI_RELU_SQ)
    src, dst = torch.randperm(T + 2, generator=g)[:T].int(), torch.randperm(T, generator=g).int()
    src_d, dst_d = src.cuda(), dst.cuda()
    y = torch.full((T, 3 * M), -7.0, device="cuda")
    B.gemm_strided(B.GemmDesc(y=y.data_ptr(), rows=T, groups=3, y_row_stride=3 * M, y_group_stride=M, x_row_index=src_d.data_ptr(),
                              y_row_index=dst_d.data_ptr(), **base))
    ref = torch.relu(torch.einsum("tk,gmk->tgm", x[src.long(), :K].double(), w[..., :K].double())) ** 2
    tol = 1e-6 * K * (1 + ref.sqrt().max())
    assert float((y.cpu().double()[dst.long()].reshape(T, 3, M) - ref).abs().max()) < tol
    expert = torch.randint(0, 3, (T, 1), generator=g, dtype=torch.int32)
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), 3)
    y = torch.full((T, M), float("nan"), device="cuda")
    B.gemm_strided(B.GemmDesc(y=y.data_ptr(), y_row_stride=M, tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(),
                              n_tiles=nt.data_ptr(), max_tiles=max_tiles, max_tile_rows=T, x_row_index=pos_row.data_ptr(), y_row_index=pos_pair.data_ptr(),
                              **base))
    ref = torch.relu(torch.einsum("tk,tmk->tm", x[:T, :K].double(), w[expert[:, 0].long(), :, :K].double())) ** 2
    assert float((y.cpu().double() - ref).abs().max()) < tol


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,d", [(1, 4), (3, 1020), (5, 1024), (300, 1028), (2, 4100)])
def test_dyt_step_starts_joins_and_picks_rows(dtype, rows, d):
    """an embedding row and its norm, a stored or routed output through the post-norm and the next norm, picked rows normed; against double
    precision: a few fp32 operations per value (tanh within 2e-6), a bf16 result rounded once"""
    from pegainfer_amd import ops_blocks as B
    g, dt = torch.Generator().manual_seed(rows + d), DT[dtype]
    st = lambda *s: torch.randn(*s, generator=g).to(dt)  # noqa: E731
    emb, ids = st(7, d), torch.randint(0, 7, (rows,), generator=g, dtype=torch.int32)
    pa, pw, pb, na, nw, nb, y = st(1), st(d), st(d), st(1), st(d), st(d), st(rows, d)
    pairs, wt = torch.randn(rows * 3, d, generator=g), torch.rand(rows, 3, generator=g)
    D64 = lambda t: t.double()  # noqa: E731
    norm = lambda t, a, w, b: torch.tanh(D64(a) * t) * D64(w) + D64(b)  # noqa: E731

    def close_(got, ref, stored):
        tol = 4e-6 * (1 + ref.abs()) + (ref.abs() * 2.0 ** -8 if stored and dtype == "bfloat16" else 0)
        assert bool(((got.cpu().double() - ref).abs() <= tol).all())
    k = {n: t.cuda() for n, t in dict(post_alpha=pa, post_w=pw, post_b=pb, next_alpha=na, next_w=nw, next_b=nb).items()}
    nxt = {n: k[n] for n in ("next_alpha", "next_w", "next_b")}
    x, out = torch.full((rows, d), float("nan"), device="cuda"), torch.zeros(rows, d, dtype=dt, device="cuda")
    ed, idd = emb.cuda(), ids.cuda()
    B.dyt_step(dt, rows, d, x=x, embed=ed, token_ids=idd, out=out, **nxt)
    ref = D64(emb)[ids.long()]
    close_(x, ref, False)
    close_(out, norm(ref, na, nw, nb), True)
    routed = (D64(wt)[:, :, None] * D64(pairs).view(rows, 3, d)).sum(1)
    for src, v in ((dict(y=y.cuda()), D64(y)), (dict(y_pairs=pairs.cuda(), weight=wt.cuda(), top=3), routed)):
        before = x.cpu().double()
        B.dyt_step(dt, rows, d, x=x, out=out, **src, **k)
        ref = before + norm(v, pa, pw, pb)
        # a routed sum is rounded as a stored one is: half a unit of it, through the post-norm's slope alpha * w
        slack = (v.abs() * 2.0 ** -8 * D64(pa).abs() * D64(pw).abs() if "y_pairs" in src and dtype == "bfloat16" else 0)
        assert bool(((x.cpu().double() - ref).abs() <= 4e-6 * (1 + ref.abs()) + slack).all())
        close_(out, norm(x.cpu().double(), na, nw, nb), True)
    before, pick = x.clone(), torch.randint(0, rows, (4,), generator=g, dtype=torch.int32).cuda()
    o4 = torch.zeros(4, d, dtype=dt, device="cuda")
    B.dyt_step(dt, 4, d, x=x, row_index=pick, out=o4, **nxt)
    close_(o4, norm(before.cpu().double()[pick.cpu().long()], na, nw, nb), True)
    assert torch.equal(x, before)


@pytest.mark.parametrize("T,ff,D,slices", [(1, 8, 8, 2), (1, 512, 1024, 0), (5, 40, 72, 3), (8, 136, 520, 1), (16, 264, 64, 2), (16, 16, 2056, 0)])
@pytest.mark.parametrize("glu", [0, 1, 2])
def test_experts_of_few_rows_with_activation_and_shared_slices(T, ff, D, slices, glu):
    """gate and up rows in one wave, an expert that all rows take in slices behind the table's columns: both products of the feed-forward against
    double precision; the first product's rows enter the second as they were stored.  Sums of D or ff products of about one in fp32."""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(T * 100 + ff + slices)
    E, top, sff, two = 6, 3, slices * ff, 2 if glu else 1
    bf = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    x, up, down, s_up, s_down = bf(T, D), bf(E, two * ff, D), bf(E, D, ff), bf(max(1, two * sff), D), bf(D, max(1, sff))
    expert = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).int()
    dev_ = [t.cuda() for t in (x, up, down, s_up, s_down)]
    xd, upd, downd, sud, sdd = dev_
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), E)
    P, n = T * top, T * top + slices * T
    act, y = torch.full((n, ff), float("nan"), device="cuda").bfloat16(), torch.full((n, D), float("nan"), device="cuda")
    table = dict(tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(), max_tiles=max_tiles, max_tile_rows=T)
    shared = dict(shared_groups=slices, shared_rows=T, shared_pos0=P)
    limit, s_limit, alpha = 9.0, 5.0, 1.702
    g1 = B.GemmDesc(x=xd.data_ptr(), w=upd.data_ptr(), y=act.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=0, m=ff, k=D, x_row_stride=D, w_m_stride=D,
                    w_k_stride=1, w_group_stride=two * ff * D, y_row_stride=ff, x_row_index=pos_row.data_ptr(), epilogue=0 if glu else B.EPI_RELU_SQ, **table)
    B.expert_rows(B.ExpertRowsDesc(g=g1, glu=glu, limit=limit, alpha=alpha, shared_limit=s_limit, shared_w=sud.data_ptr() if slices else None,
                                   shared_m_stride=D, shared_group_stride=ff * D, shared_up=sff * D, **shared))
    g2 = B.GemmDesc(x=act.data_ptr(), w=downd.data_ptr(), y=y.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=1, m=D, k=ff, x_row_stride=ff, w_m_stride=ff,
                    w_k_stride=1, w_group_stride=D * ff, y_row_stride=D, y_row_index=pos_pair.data_ptr(), **table)
    B.expert_rows(B.ExpertRowsDesc(g=g2, shared_w=sdd.data_ptr() if slices else None, shared_m_stride=sff, shared_group_stride=ff, **shared))

    def f(z, lim):
        if not glu:
            return torch.relu(z) ** 2
        a, u = z.chunk(2, -1)
        if glu == 1:
            return a * torch.sigmoid(a) * u
        a, u = a.clamp(max=lim), u.clamp(-lim, lim)
        return a * torch.sigmoid(alpha * a) * (u + 1)
    at = pos_pair.cpu().long()                       # sorted position -> pair
    want = torch.stack([f(x[p // top].double() @ up[expert.view(-1)[p]].double().T, limit) for p in at.tolist()])
    if slices:
        s = f(x.double() @ s_up.double().T, s_limit)
        want = torch.cat([want] + [s[:, j * ff:(j + 1) * ff] for j in range(slices)])
    a = act.cpu().double()
    assert float(((a - want).abs() / (want.abs() * 2.0 ** -8 + 1e-6 * D * (1 + want.abs().max().sqrt()))).max()) <= 1.0
    rows = torch.full((n, D), float("nan"), dtype=torch.float64)
    for q, p in enumerate(at.tolist()):
        rows[p] = a[q] @ down[expert.view(-1)[p]].double().T
    for j in range(slices):
        rows[P + j * T:P + (j + 1) * T] = a[P + j * T:P + (j + 1) * T] @ s_down[:, j * ff:(j + 1) * ff].double().T
    assert float((y.cpu().double() - rows).abs().max()) <= 1e-6 * ff * float(a.abs().max().clamp(min=1))
    if slices:
        w, gate = torch.rand(T, top, generator=g), torch.randn(T, generator=g)
        got = B.route_combine_pairs(y[:P], w.cuda(), y[P:].view(slices, T, D), gate.cuda(), torch.float32)
        ref = torch.einsum("tc,tcd->td", w.double(), rows[:P].view(T, top, D)) + torch.sigmoid(gate.double())[:, None] * rows[P:].view(slices, T, D).sum(0)
        assert float((got.cpu().double() - ref).abs().max()) <= 2e-6 * ff * float(a.abs().max().clamp(min=1))


@pytest.mark.parametrize("xd,yd", [("bfloat16", "bfloat16"), ("bfloat16", "float32"), ("float32", "bfloat16"), ("float32", "float32")])
@pytest.mark.parametrize("T,M,K,G", [(17, 128, 8, 1), (65, 130, 56, 2), (128, 127, 64, 3), (129, 300, 72, 1), (200, 1, 200, 2), (513, 514, 136, 40)])
def test_tiles_on_the_matrix_cores_at_their_edges(T, M, K, G, xd, yd):
    """slices that end inside K (what lies behind K in the wider rows is no number), rows and outputs past a tile's end, several groups, odd output
    rows, gathered and scattered rows with a gate: against the product of the operands as the matrix cores see them (fp32 rows rounded to
    bf16).  Sums of K products of about one in fp32: 1e-6 K; a bf16 result adds half a unit in the last place, 2^-8 of the value."""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(T + M)
    xs, ws = G * (K + 8) + 8, K + 16
    x = torch.full((T + 3, xs), float("nan"))
    w = torch.full((G, M, ws), float("nan"))
    for i in range(G):
        x[:, i * (K + 8):i * (K + 8) + K] = torch.randn(T + 3, K, generator=g)
    w[:, :, :K] = C.bf16_round(torch.randn(G, M, K, generator=g))
    if xd == "bfloat16":
        x = C.bf16_round(x)
    src, dst = torch.randperm(T + 3, generator=g)[:T].int(), torch.randperm(T, generator=g).int()
    gate = torch.randn(T + 3, G, generator=g)
    x_d, w_d, src_d, dst_d, gate_d = dev(x, DT[xd]), dev(w, torch.bfloat16), src.cuda(), dst.cuda(), gate.cuda()
    ref = torch.einsum("tgk,gmk->tgm", C.bf16_round(x[src.long()]).double()[:, :G * (K + 8)].reshape(T, G, K + 8)[..., :K], w[..., :K].double())
    for epi in (B.EPI_NONE, B.EPI_RELU_SQ, B.EPI_SIGMOID_GATE):
        r = ref if epi == B.EPI_NONE else torch.relu(ref) ** 2 if epi == B.EPI_RELU_SQ else ref * torch.sigmoid(gate[src.long()].double())[..., None]
        for pad in (0, 1):
            y = torch.full((T, G * M + pad), -7.0, device="cuda", dtype=DT[yd])
            B.gemm_strided(B.GemmDesc(x=x_d.data_ptr(), w=w_d.data_ptr(), y=y.data_ptr(), x_dtype=B._dt(x_d), w_dtype=0, y_dtype=B._dt(y), m=M, k=K,
                                      rows=T, groups=G, x_row_stride=xs, x_group_stride=K + 8, w_m_stride=ws, w_k_stride=1, w_group_stride=M * ws,
                                      y_row_stride=G * M + pad, y_group_stride=M, x_row_index=src_d.data_ptr(), y_row_index=dst_d.data_ptr(),
                                      epilogue=epi, gate=gate_d.data_ptr(), gate_dtype=1, gate_row_stride=G))
            got = y.cpu().double()
            assert pad == 0 or float((got[:, -1] + 7.0).abs().max()) == 0.0
            got = got[dst.long()][:, :G * M].reshape(T, G, M)
            tol = 1e-6 * K * (1 + r.abs()) ** (1 if epi != B.EPI_RELU_SQ else 0.5) * (4 if epi == B.EPI_RELU_SQ else 1)
            assert bool(((got - r).abs() <= tol + (r.abs() / 256 if yd == "bfloat16" else 0)).all()), (epi, pad, float((got - r).abs().max()))


@pytest.mark.parametrize("rows_per_tile", [64, 128])
def test_tiles_of_an_expert_table_reach_every_pair(rows_per_tile):
    """live tiles dealt over eight runs: one tile, seven, eight, nine and many, more places in the table than tiles"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(rows_per_tile)
    for E, rows, top in ((1, 20, 1), (7, 40, 2), (8, 64, 3), (9, 41, 4), (40, 300, 5)):
        K, M = 72, 200
        expert = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(rows)]).int()
        pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), E, rows_per_tile=rows_per_tile)
        x, w = C.bf16_round(torch.randn(rows, K, generator=g)), C.bf16_round(torch.randn(E, M, K, generator=g))
        xd, wd = dev(x, torch.bfloat16), dev(w, torch.bfloat16)
        y = torch.full((rows * top, M), float("nan"), device="cuda")
        B.gemm_strided(B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=1, m=M, k=K, x_row_stride=K,
                                  w_m_stride=K, w_k_stride=1, w_group_stride=M * K, y_row_stride=M, tile_group=tg.data_ptr(),
                                  tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(), max_tiles=max_tiles,
                                  x_row_index=pos_row.data_ptr(), y_row_index=pos_pair.data_ptr(), tile_rows_cap=rows_per_tile))
        ref = torch.einsum("pk,pmk->pm", x.double().repeat_interleave(top, 0), w.double()[expert.reshape(-1).long()])
        assert float((y.cpu().double() - ref).abs().max()) < 1e-6 * K * (1 + float(ref.abs().max()))


@pytest.mark.parametrize("known", [1, 4, 16, 0])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_empty_tiles_of_a_table_are_passed_over(dtype, known):
    """a tile without rows, before the first position, between others and at the end: nothing is read or written for it"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(known)
    T, M, K = min(known or 40, 5), 70, 72
    x, w = C.bf16_round(torch.randn(T, K, generator=g)), C.bf16_round(torch.randn(3, M, K, generator=g))
    xd, wd = dev(x, DT[dtype]), dev(w, DT[dtype])
    tg, t0, tr, nt = (torch.tensor(v, dtype=torch.int32).cuda() for v in ([2, 0, 1, 1], [0, 0, T, T], [0, T, 0, 0], [4]))
    rows = torch.arange(T, dtype=torch.int32).flip(0).contiguous()
    rd = rows.cuda()
    y = torch.full((T, M), -7.0, device="cuda")
    B.gemm_strided(B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=B._dt(xd), w_dtype=B._dt(wd), y_dtype=1, m=M, k=K, x_row_stride=K,
                              w_m_stride=K, w_k_stride=1, w_group_stride=M * K, y_row_stride=M, tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(),
                              tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(), max_tiles=4, max_tile_rows=known, x_row_index=rd.data_ptr()))
    ref = x.double()[rows.long()] @ w[0].double().T
    assert float((y.cpu().double() - ref).abs().max()) < 1e-6 * K * (1 + float(ref.abs().max()))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_strided_gemm_forms_agree(dtype):
    """the few-rows form (<= 8 rows), the matrix-core tile form (bf16 weights) and the fp32-FMA tile form compute the same
    products of the stored values; only the order of the fp32 sums differs"""
    from pegainfer_amd import ops_blocks as B
    td = DT[dtype]
    g = torch.Generator().manual_seed(7)
    for (T, M, K) in [(1, 96, 128), (4, 33, 256), (7, 40, 64), (8, 200, 1024), (9, 40, 64), (70, 130, 192), (64, 64, 64), (200, 72, 320)]:
        x, w = C.bf16_round(torch.randn(T, K, generator=g)), C.bf16_round(torch.randn(M, K, generator=g))
        ref = x.double() @ w.double().T
        for epi in (B.EPI_NONE, B.EPI_RELU_SQ):
            want = ref if epi == B.EPI_NONE else torch.relu(ref) ** 2
            fast = B.linear(dev(x, td), dev(w, td), out_dtype=torch.float32, epilogue=epi).cpu()
            plain = B.linear(dev(x, td), dev(w, td), out_dtype=torch.float32, epilogue=epi, plain=True).cpu()
            tol = 2e-5 * K * (1 if epi == B.EPI_NONE else 10)
            assert (fast.double() - want).abs().max() < tol and (plain.double() - want).abs().max() < tol, (T, M, K, epi)
    # grouped rows with a small bound on the rows per tile: the few-rows form walks the same tile table
    rows, top, E, d, ff = 5, 2, 6, 64, 24
    expert = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(rows)]).int()
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), E)
    x, w = C.bf16_round(torch.randn(rows, d, generator=g)), C.bf16_round(torch.randn(E, ff, d, generator=g))
    xd, wd = dev(x, td), dev(w, td)
    outs = []
    for plain in (0, 1):
        y = torch.zeros(rows * top, ff, device="cuda")
        B.gemm_strided(B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=B._dt(xd), w_dtype=B._dt(wd), y_dtype=1,
                                  m=ff, k=d, x_row_stride=d, w_m_stride=d, w_k_stride=1, w_group_stride=ff * d, y_row_stride=ff,
                                  tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(),
                                  max_tiles=max_tiles, x_row_index=pos_row.data_ptr(), y_row_index=pos_pair.data_ptr(),
                                  max_tile_rows=rows, plain=plain))
        outs.append(y.cpu())
    ref = torch.einsum("pd,pfd->pf", x.double().repeat_interleave(top, 0), w.double()[expert.reshape(-1).long()])
    assert (outs[0].double() - ref).abs().max() < 1e-4 and (outs[1].double() - ref).abs().max() < 1e-4


@pytest.mark.parametrize("x_type", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,M,K", [(1, 16, 8), (2, 33, 72), (3, 48, 200), (16, 17, 256), (5, 100, 520), (15, 64, 512), (9, 31, 2056),
                                   (8, 40000, 64), (16, 20011, 136), (17, 40, 64)])
def test_few_rows_on_the_matrix_cores(T, M, K, x_type):
    """Row counts up to the form's sixteen and the first beyond, outputs that are no multiple of a block of 16, k that ends inside a piece of 64,
    one, two and four waves per block, one and two blocks per wave.  Products are exact (an fp32 x is not rounded: parts of it sum to it), so
    the error is that of fp32 sums: half an ulp of the running sum per addition, at most K / 2 of them in a row."""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(T * 1000 + K)
    x, w = torch.randn(T, K, generator=g), C.bf16_round(torch.randn(M, K, generator=g))
    x[0, :4] *= 2.0 ** 60                       # far apart: the small parts must not reach the large row's neighbours
    if x_type == torch.bfloat16 or T > 16:      # the tile form that takes over beyond 16 rows rounds an fp32 x
        x = C.bf16_round(x)
    got = B.linear(x.to(x_type).cuda(), w.bfloat16().cuda(), out_dtype=torch.float32).cpu().double()
    scale = x.double().abs() @ w.double().abs().T
    assert ((got - x.double() @ w.double().T).abs() <= (K / 2 + 16) * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("T,M,K", [(9, 1, 8), (32, 64, 64), (33, 63, 72), (64, 65, 136), (65, 17, 1032), (130, 4200, 64), (4200, 130, 40)])
def test_fp32_tiles_on_the_matrix_cores(T, M, K):
    """32- and 64-row tiles, rows and outputs that end inside a tile, k that ends inside a slice of 64; fp32 products and sums: at most K / 4
    additions of four products each in a row, half an ulp of the running sum per addition and product."""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(T + M + K)
    x, w = torch.randn(T, K, generator=g), torch.randn(M, K, generator=g)
    got = B.linear(x.cuda(), w.cuda(), out_dtype=torch.float32).cpu().double()
    bound = (K + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((got - x.double() @ w.double().T).abs() <= bound).all()


def test_fp32_tiles_over_a_tile_table():
    """gathered rows, a table whose last tile of an expert is partly filled, outputs scattered by pair"""
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(5)
    rows, top, E, d, ff = 150, 2, 3, 72, 100
    expert = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(rows)]).int()
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), E)
    x, w = torch.randn(rows, d, generator=g), torch.randn(E, ff, d, generator=g)
    xd, wd, y = x.cuda(), w.cuda(), torch.zeros(rows * top, ff, device="cuda")
    B.gemm_strided(B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=1, w_dtype=1, y_dtype=1, m=ff, k=d, x_row_stride=d,
                              w_m_stride=d, w_k_stride=1, w_group_stride=ff * d, y_row_stride=ff, tile_group=tg.data_ptr(),
                              tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(), max_tiles=max_tiles,
                              x_row_index=pos_row.data_ptr(), y_row_index=pos_pair.data_ptr()))
    ref = torch.bmm(x.double().repeat_interleave(top, 0)[:, None], w.double()[expert.reshape(-1).long()].transpose(1, 2).contiguous())[:, 0]
    assert (y.cpu().double() - ref).abs().max() < (d + 8) * 2.0 ** -24 * d * 16


def test_few_rows_keep_infinities():
    from pegainfer_amd import ops_blocks as B
    x, w = torch.ones(3, 64), torch.ones(16, 64)
    x[0, 5], x[1, 7], x[2, 9] = float("inf"), float("nan"), 3.4e38
    got = B.linear(x.cuda(), w.bfloat16().cuda(), out_dtype=torch.float32).cpu()
    assert torch.isinf(got[0]).all() and torch.isnan(got[1]).all() and torch.isfinite(got[2]).all()


@pytest.mark.parametrize("bits", [0x7F800001, 0xFF80FFFF, 0x7F810000, 0xFFFFFFFF])
def test_few_rows_keep_what_is_no_number(bits):
    """whatever the payload, also one that lies in the bits a bf16 does not have"""
    from pegainfer_amd import ops_blocks as B
    x, w = torch.ones(3, 72), torch.ones(17, 72)
    x.view(torch.int32)[1, 70] = np.uint32(bits).astype(np.int32).item()
    got = B.linear(x.cuda(), w.bfloat16().cuda(), out_dtype=torch.float32).cpu()
    assert torch.isnan(got[1]).all() and torch.equal(got[0], got[2]) and float(got[0, 0]) == 72.0


@pytest.mark.parametrize("M", [19, 40003])
def test_few_rows_against_infinite_weights(M):
    """finite values times an infinite weight are infinities of their sign, whether a bf16 holds the value or not; zeros and infinities of both signs
    give no number"""
    from pegainfer_amd import ops_blocks as B
    x, w = torch.full((6, 136), 0.7), torch.full((M, 136), 0.5)
    x[0, 5], x[1, 5], x[2, 5], x[3, 5], x[4, 5] = 1.5, -0.3, 0.0, float("inf"), float("-inf")
    w[1, 5], w[2, 5] = float("inf"), float("-inf")
    w[M - 1, 5], w[M - 1, 130] = float("inf"), float("-inf")
    got = B.linear(x.cuda(), w.bfloat16().cuda(), out_dtype=torch.float32).cpu().double()
    ref = torch.tensor([[sum((x[r].double() * w[m].double()).tolist()) for m in (0, 1, 2, M - 1)] for r in range(6)], dtype=torch.float64)
    torch.testing.assert_close(got[:, [0, 1, 2, M - 1]], ref, rtol=1e-5, atol=1e-4, equal_nan=True)


def test_grouped_gemm_over_128_row_tiles():
    from pegainfer_amd import ops_blocks as B
    g = torch.Generator().manual_seed(11)
    rows, top, E, d, ff = 400, 2, 3, 64, 136         # ~267 pairs per expert: two full 128-row tiles and a part of a third
    expert = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(rows)]).int()
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), E, rows_per_tile=128)
    assert int(tr.cpu()[:int(nt.item())].max()) == 128
    x, w = C.bf16_round(torch.randn(rows, d, generator=g)), C.bf16_round(torch.randn(E, ff, d, generator=g))
    xd, wd = dev(x, torch.bfloat16), dev(w, torch.bfloat16)
    y = torch.zeros(rows * top, ff, device="cuda")
    B.gemm_strided(B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=1, m=ff, k=d,
                              x_row_stride=d, w_m_stride=d, w_k_stride=1, w_group_stride=ff * d, y_row_stride=ff,
                              tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(), n_tiles=nt.data_ptr(),
                              max_tiles=max_tiles, x_row_index=pos_row.data_ptr(), y_row_index=pos_pair.data_ptr(),
                              tile_rows_cap=128))
    ref = torch.einsum("pd,pfd->pf", x.double().repeat_interleave(top, 0), w.double()[expert.reshape(-1).long()])
    assert (y.cpu().double() - ref).abs().max() < 1e-4
    with pytest.raises(RuntimeError):                 # the 64-row fp32-FMA form refuses a table cut for 128-row tiles
        B.gemm_strided(B.GemmDesc(x=xd.data_ptr(), w=wd.data_ptr(), y=y.data_ptr(), x_dtype=0, w_dtype=0, y_dtype=1, m=ff, k=d,
                                  x_row_stride=d, w_m_stride=d, w_k_stride=1, w_group_stride=ff * d, y_row_stride=ff,
                                  tile_group=tg.data_ptr(), tile_row0=t0.data_ptr(), tile_rows=tr.data_ptr(),
                                  n_tiles=nt.data_ptr(), max_tiles=max_tiles, x_row_index=pos_row.data_ptr(),
                                  y_row_index=pos_pair.data_ptr(), tile_rows_cap=128, plain=1))
