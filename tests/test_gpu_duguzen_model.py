"""The Duguzen engine (host runtime, latent cache, batched step, scheduler) on the GPU against the plain restatement
(oracle/duguzen_ref.py) on small random models: whole prompts, prefill against token-by-token decoding, portions down to
two tokens, unequal requests in one batch against each alone, pages and slots that are freed and used again, long decoding
across the attention's key split, a checkpoint folder through the registry, and greedy generation through the scheduler."""
import json
import os

import numpy as np
import pytest
import torch

import duguzen_common as C

pytestmark = pytest.mark.gpu

CONFIGS = {"a": C.config_a, "b": C.config_b, "tiny": C.config_tiny, "odd": C.config_odd}


def check(got, ref, dtype, what=""):
    """fp32: every row inside the tolerance.  bf16: random routers have near ties, and a bf16 rounding that flips one expert
    choice moves that row (and the rows that attend to it) by far more than rounding - so nine rows in ten must be inside
    the rounding tolerance and none may be wrong outright; a fault that hits single rows is the fp32 run's to find."""
    e = C.row_err(got, ref)
    if dtype == "float32" or len(e) < 4:
        assert e.max() < (C.TOL[dtype] if dtype == "float32" else 0.5), (what, float(e.max()), int(e.argmax()))
    else:
        assert np.quantile(e, 0.9) < C.TOL[dtype] and e.max() < 0.5, (what, float(np.quantile(e, 0.9)), float(e.max()))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["a", "b", "odd", "tiny"])
def test_whole_prompt_every_position_and_every_layer(name, dtype):
    cfg = CONFIGS[name]()
    w = C.random_weights(cfg, 11)
    toks = C.tokens_for(cfg, 70, 1)
    taps = []
    ref = C.oracle_logits(cfg, w, toks, taps)
    eng = C.engine_for(cfg, w, dtype)
    eng.debug_hidden_enable(True)
    r = eng.new_request()
    got = eng.step([(r, toks)], want=list(range(len(toks))))
    check(got, ref, dtype)
    H = eng.debug_hidden(len(toks))
    for i, t in enumerate(taps):
        scale = float(t.abs().max())
        per_row = np.abs(H[i] - t.numpy()).max(-1) / scale
        if dtype == "float32":
            assert per_row.max() < 2e-5, i
        else:                        # a flipped expert choice moves single rows (see check)
            assert np.quantile(per_row, 0.85) < 4e-2, (i, float(np.quantile(per_row, 0.85)))
    if dtype == "bfloat16":          # the tuned GEMM routes and the plain tile kernel agree to rounding
        eng.drop_request(r)
        eng.set_plain_kernels(True)
        r = eng.new_request()
        check(eng.step([(r, toks)], want=list(range(len(toks)))), ref, dtype)
    eng.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["a", "odd"])
def test_prefill_then_token_by_token(name, dtype):
    cfg = CONFIGS[name]()
    w = C.random_weights(cfg, 12)
    toks = C.tokens_for(cfg, 60, 2)
    ref = C.oracle_logits(cfg, w, toks)
    eng = C.engine_for(cfg, w, dtype)
    r = eng.new_request()
    rows = [eng.step([(r, toks[:15])], want=list(range(15)))]          # 15: the prompt ends one short of a page
    for t in range(15, 60):
        rows.append(eng.step([(r, [toks[t]])]))
    check(np.concatenate(rows), ref, dtype)
    r2 = eng.new_request()                                               # the very first tokens decoded one by one, too
    first = np.concatenate([eng.step([(r2, [toks[t]])]) for t in range(4)])
    check(first, ref[:4], dtype)
    eng.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("sizes", [[2, 3, 1, 17, 16, 2, 29], [31, 2, 2, 33, 2], [16, 16, 16, 16, 6]])
def test_portions(dtype, sizes):
    cfg = C.config_a()
    w = C.random_weights(cfg, 13)
    toks = C.tokens_for(cfg, sum(sizes), 3)
    ref = C.oracle_logits(cfg, w, toks)
    eng = C.engine_for(cfg, w, dtype)
    r, at, rows = eng.new_request(), 0, []
    for n in sizes:
        rows.append(eng.step([(r, toks[at:at + n])], want=list(range(n))))
        at += n
    got = np.concatenate(rows)
    check(got, ref, dtype)
    if dtype == "float32":           # cutting the prompt changes nothing at all in the fp32 engine: same kernels, same k order
        r2 = eng.new_request()
        whole = eng.step([(r2, toks)], want=list(range(len(toks))))
        assert np.abs(whole - got).max() <= 1e-5 * np.abs(whole).max()
    eng.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_unequal_requests_in_one_batch_against_each_alone(dtype):
    cfg = C.config_a()
    w = C.random_weights(cfg, 14)
    P = [C.tokens_for(cfg, n, 10 + n) for n in (37, 5, 50, 1)]
    refs = [C.oracle_logits(cfg, w, p) for p in P]
    eng = C.engine_for(cfg, w, dtype, max_tokens=256)
    ids = [eng.new_request() for _ in P]
    # schedule: (request, tokens taken) per step - portions of some beside single tokens of others; a request sits a step out
    plan = [[(0, 20), (1, 2), (3, 1)], [(0, 2), (1, 1), (2, 33)], [(0, 1), (2, 1)], [(0, 14), (1, 2), (2, 16)]]
    at, got = [0] * 4, [[] for _ in P]
    for stp in plan:
        entries, want, off = [], [], 0
        for q, n in stp:
            entries.append((ids[q], P[q][at[q]:at[q] + n]))
            want += list(range(off, off + n))
            off += n
        lg = eng.step(entries, want=want)
        off = 0
        for q, n in stp:
            got[q].append(lg[off:off + n])
            at[q] += n
            off += n
    alone = C.engine_for(cfg, w, dtype, max_tokens=256)
    for q in range(4):
        g = np.concatenate(got[q])
        check(g, refs[q][:at[q]], dtype, q)
        r = alone.new_request()
        solo = alone.step([(r, P[q][:at[q]])], want=list(range(at[q])))
        alone.drop_request(r)
        if dtype == "float32":       # what else is in the batch does not reach a row's arithmetic
            assert np.abs(solo - g).max() <= 1e-5 * np.abs(solo).max(), q
    eng.close()
    alone.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_pages_and_slots_are_used_again(dtype):
    cfg = C.config_b()
    w = C.random_weights(cfg, 15)
    eng = C.engine_for(cfg, w, dtype, max_tokens=96, max_requests=2)      # 6 pages of 16 tokens, 2 slots
    assert eng.capacity_pages() == 6
    A, B_, Cq, Dq = (C.tokens_for(cfg, n, 20 + n) for n in (40, 50, 30, 33))
    a = eng.new_request()
    check(eng.step([(a, A)], want=list(range(40))), C.oracle_logits(cfg, w, A), dtype)        # 3 pages
    b = eng.new_request()
    with pytest.raises(RuntimeError):
        eng.new_request()                                                                       # both slots are taken
    with pytest.raises(RuntimeError):
        eng.step([(b, B_)])                                                                     # 4 pages wanted, 3 free
    assert eng.seq_len(b) == 0 and eng.available_pages() == 3 and eng.seq_len(a) == 40         # a rejected step changes nothing
    eng.drop_request(a)
    assert eng.available_pages() == 6
    check(eng.step([(b, B_)], want=list(range(50))), C.oracle_logits(cfg, w, B_), dtype)       # reuses a's pages
    c = eng.new_request()                                                                       # reuses a's slot
    lg = eng.step([(c, Cq[:20]), (b, B_[:0] + [B_[0]])], want=list(range(20)))                 # b decodes on while c starts
    check(lg, C.oracle_logits(cfg, w, Cq)[:20], dtype)
    eng.drop_request(b)
    d = eng.new_request()
    lg = eng.step([(d, Dq), (c, Cq[20:])], want=list(range(33 + 10)))
    check(lg[:33], C.oracle_logits(cfg, w, Dq), dtype)
    check(lg[33:], C.oracle_logits(cfg, w, Cq)[20:], dtype)
    eng.close()


def test_long_decoding_across_the_key_split():
    cfg = C.config_tiny()
    w = C.random_weights(cfg, 16)
    toks = C.tokens_for(cfg, 1060, 4)
    ref = C.oracle_logits(cfg, w, toks)
    eng = C.engine_for(cfg, w, "float32", max_tokens=1100)
    r = eng.new_request()
    got = [eng.step([(r, toks[:1000])], want=[0, 1, 255, 256, 999])]
    for t in range(1000, 1060):       # positions 1023 / 1024: the last key of one split, the first of the next
        got.append(eng.step([(r, [toks[t]])]))
    check(np.concatenate(got), ref[[0, 1, 255, 256, 999] + list(range(1000, 1060))], "float32")
    eng.close()


@pytest.mark.parametrize("dtype,name", [("bfloat16", "a"), ("float32", "b"), ("bfloat16", "odd")])
def test_replayed_decode_steps_give_what_eager_ones_give(dtype, name):
    """Decode steps are replayed from graphs, one per batch and context length rounded up to 256 tokens; the per-layer tap turns that off.  The
    same bits either way: contexts of unequal length that cross the rounding, other steps between the replays, buffers that grow."""
    cfg = CONFIGS[name]()
    w = C.random_weights(cfg, 31)
    engs = [C.engine_for(cfg, w, dtype, max_tokens=1200, max_requests=4) for _ in range(2)]
    engs[1].debug_hidden_enable(True)
    out = []
    for eng in engs:
        r, got = [eng.new_request() for _ in range(3)], []
        toks = C.tokens_for(cfg, 400, 7)
        for i, n in enumerate((250, 17, 240)):
            got.append(eng.step([(r[i], toks[:n])]))
        for t in range(20):
            use = r if t % 5 else r[:1]                     # two batch sizes in turn
            lg, tk = eng.step([(q, [toks[300 + t]]) for q in use], tokens=True)
            got += [lg, tk]
            if t == 12:
                late = eng.new_request()
                got.append(eng.step([(late, toks[:200])], want=list(range(60))))      # more rows and more wanted rows than before
                eng.drop_request(late)
        out.append(got)
        eng.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_more_shapes_than_graphs_are_kept_and_contexts_past_the_last_graph():
    """80 shapes of a decode step (1 - 8 requests, any number of wanted rows, tokens or not) twice in turn, more than the 64 graphs that are kept; then a
    context that grows from the last one captured (8192 tokens) to one that runs eagerly.  The same bits as steps that are never captured."""
    cfg = C.config_tiny()
    w = C.random_weights(cfg, 5)
    engs = [C.engine_for(cfg, w, "bfloat16", max_tokens=9000, max_requests=8) for _ in range(2)]
    engs[1].debug_hidden_enable(True)
    toks = C.tokens_for(cfg, 8220, 9)
    shapes = [(n, k, t) for n in range(1, 9) for k in range(n + 1) for t in ((False, True) if k else (False,))]
    assert len(shapes) == 80
    out = []
    for eng in engs:
        r, got = [eng.new_request() for _ in range(8)], []
        eng.step([(q, toks[i:i + 3 + 5 * i]) for i, q in enumerate(r)], want=[])
        for step, (n, k, t) in enumerate(shapes + shapes):
            res = eng.step([(q, [toks[step]]) for q in r[:n]], want=list(range(k)), logits=k > 0, tokens=t)
            got += [] if not k else list(res) if t else [res]
        for q in r[1:]:
            eng.drop_request(q)
        done = eng.seq_len(r[0])
        eng.step([(r[0], toks[done:8180])], want=[])
        for t in range(8180, 8210):
            got.append(eng.step([(r[0], [toks[t]])]))
        assert eng.seq_len(r[0]) == 8210
        out.append(got)
        eng.close()
    assert len(out[0]) == len(out[1]) and all(np.array_equal(a, b) for a, b in zip(*out))


def test_checkpoint_folder_through_the_registry_and_trace_replay(tmp_path):
    from safetensors.torch import save_file
    from pegainfer_amd import registry
    cfg = C.config_b()
    w = C.random_weights(cfg, 17)
    json.dump(cfg, open(tmp_path / "config.json", "w"))
    save_file({k: v.bfloat16().contiguous() for k, v in w.items()}, str(tmp_path / "model.safetensors"))
    assert registry.family_of(cfg) == "duguzen"
    toks = C.tokens_for(cfg, 25, 5)
    ref = C.oracle_logits(cfg, w, toks)
    for dtype in ("bfloat16", "float32"):
        eng = registry.load_engine(str(tmp_path), dtype=dtype, max_tokens=64, max_requests=2)
        r = eng.new_request()
        check(eng.step([(r, toks)], want=list(range(25))), ref, dtype)
        eng.close()
    with pytest.raises(ValueError):
        registry.load_engine(str(tmp_path), dtype="float16")
    # the trace replay program: two requests, portions, a request that ends and frees its slot
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    steps = [{"step": 0, "entries": [{"id": "x", "tokens": toks[:7], "want": [6]}, {"id": "y", "tokens": toks[:2], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "x", "tokens": toks[7:25], "want": [0, 17]}], "end": ["x"]},
             {"step": 2, "entries": [{"id": "y", "tokens": toks[2:3], "want": [0]}], "end": ["y"]}]
    out = tmp_path / "out"
    p = subprocess.run([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", str(tmp_path), "--dtype", "float32",
                        "--out", str(out), "--max-tokens", "64"], input="\n".join(json.dumps(s) for s in steps) + "\n",
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-2000:]
    assert [l for l in p.stdout.split("\n") if l.startswith("done")] == ["done 0", "done 1", "done 2"]
    V = cfg["vocab"]
    check(np.fromfile(out / "0.f32", dtype="<f4").reshape(-1, V), ref[[6]], "float32")
    check(np.fromfile(out / "1.f32", dtype="<f4").reshape(-1, V), ref[[7, 24]], "float32")
    check(np.fromfile(out / "2.f32", dtype="<f4").reshape(-1, V), ref[[2]], "float32")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_greedy_generation_through_the_scheduler(dtype):
    from pegainfer_amd import registry
    from pegainfer_amd import scheduler as S
    cfg = C.config_a()
    w = C.random_weights(cfg, 18)
    prompts = [C.tokens_for(cfg, n, 30 + n) for n in (9, 21, 4)]
    eng = C.engine_for(cfg, w, dtype, max_tokens=256, max_requests=4)
    sch = registry.scheduler_for(eng)
    rids = [sch.submit(p, 6, params=(0.0, -1, 1.0, True)) for p in prompts]
    out = {r: [] for r in rids}
    for _ in range(40):
        if sch.step() == 0 and sch.num_active() == 0 and sch.num_deferred() == 0:
            break
        for ev in sch.poll():
            if ev[1] == S.TOKEN:
                out[ev[0]].append(int(ev[2]))
    assert all(len(v) == 6 for v in out.values()), out
    for rid, p in zip(rids, prompts):
        seq = list(p)
        for tok in out[rid]:
            lg = C.oracle_logits(cfg, w, seq)[-1]
            best = int(lg.argmax())
            margin = float(lg[best] - np.partition(lg, -2)[-2])
            if tok != best:       # only a near tie may differ, and then the engine's choice must be that runner-up
                assert margin < (1e-3 if dtype == "float32" else 0.15) and lg[tok] >= lg[best] - (1e-3 if dtype == "float32" else 0.15)
            seq.append(tok)
    assert eng.available_pages() == eng.capacity_pages()          # finished requests gave their pages back
    sch.close()
    eng.close()


def test_command_line_generates_like_the_plain_restatement(tmp_path):
    import subprocess
    import sys
    from safetensors.torch import save_file
    cfg = C.config_tiny()
    w = C.random_weights(cfg, 19)
    json.dump(cfg, open(tmp_path / "config.json", "w"))
    save_file({k: v.bfloat16().contiguous() for k, v in w.items()}, str(tmp_path / "model.safetensors"))
    prompt = C.tokens_for(cfg, 11, 6)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-m", "pegainfer_amd", "generate", "--model", str(tmp_path), "--dtype", "float32",
                        "--prompt-ids", ",".join(map(str, prompt)), "--max-new-tokens", "5"], cwd=root, capture_output=True,
                       text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-2000:]
    got = json.loads([l for l in p.stdout.split("\n") if l.startswith("{")][-1])["tokens"]
    seq = list(prompt)
    for tok in got:
        lg = C.oracle_logits(cfg, w, seq)[-1]
        assert tok == int(lg.argmax()) or lg[tok] >= lg.max() - 1e-3
        seq.append(tok)
    assert len(got) == 5


def test_a_layer_that_borrows_from_a_borrowing_layer():
    cfg = C.config_a()
    cfg["layers"].append({**cfg["layers"][2], "weights_of": 2})      # layer 5 -> layer 2 -> layer 0, with a cache of its own
    w = C.random_weights(cfg, 21)
    toks = C.tokens_for(cfg, 40, 7)
    ref = C.oracle_logits(cfg, w, toks)
    eng = C.engine_for(cfg, w, "float32")
    assert eng.layer_runs == 6
    r = eng.new_request()
    got = np.concatenate([eng.step([(r, toks[:33])], want=list(range(33))), eng.step([(r, toks[33:])], want=list(range(7)))])
    check(got, ref, "float32")
    eng.close()
