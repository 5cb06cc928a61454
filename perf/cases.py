"""Performance cases: what a user of this framework has it do, through the engines a model folder opens.

Every case serves a batch of requests once: the prompts go in (in one step or in portions), then every request is continued token by
token with tokens that are given - the replay of a trace, so that a pass does the same work and gives the same numbers every time it is
run.  Every step's greedy tokens are asked for (and, where the case samples, a sampled one), as a server does.  Outputs: the logits behind
the prompts and those of the last step, which read everything that the steps between left in the caches and states.  The tokens are no
outputs: the largest logits of a random model lie closer together than a rounding moves them.

Sizes are those of the repository's own benchmark configurations.  Qwen3-4B / 8B run at full depth, the Qwen3.5-4B hybrid with two rounds of
its layer pattern (at full depth a random hybrid turns bf16 roundings into a tenth of its logits); the other families at their benchmark's
layer sizes with one round of their layer pattern (every kind of layer once or twice).

Weights are random.  The Qwen engines make them on the device from a seed, `exact` draws the same numbers again; the other families load a
checkpoint of tensors drawn here.
"""
import functools
import math

import numpy as np
import torch
import torch.nn.functional as Fn

from pegainfer_amd import bench_duguzen, bench_feruzen, bench_kukulorn, bench_ramalix, bench_sopanex, bench_zofadra
from pegainfer_amd.duguzen import DuguzenEngine
from pegainfer_amd.feruzen import FeruzenEngine
from pegainfer_amd.kukulorn import KukulornEngine
from pegainfer_amd.qwen3 import QWEN3_4B, QWEN3_8B, Qwen3Engine
from pegainfer_amd.qwen35 import QWEN35_4B, Qwen35Engine
from pegainfer_amd.ramalix import RamalixEngine
from pegainfer_amd.sopanex import SopanexEngine
from pegainfer_amd.zofadra import ZofadraEngine

F64 = torch.float64
QWEN = {"qwen3-4b": QWEN3_4B, "qwen3-8b": QWEN3_8B, "qwen3.5-4b": QWEN35_4B}
# engine, benchmark sizes, configuration, layers kept of the benchmark's list
FAMILY = {
    "duguzen": (DuguzenEngine, bench_duguzen.SIZES, bench_duguzen.duguzen_config, 4),
    "feruzen": (FeruzenEngine, bench_feruzen.SIZES, bench_feruzen.feruzen_config, 4),
    "ramalix": (RamalixEngine, bench_ramalix.SIZES, bench_ramalix.ramalix_config, 4),
    "kukulorn": (KukulornEngine, bench_kukulorn.SIZES, bench_kukulorn.kukulorn_config, 4),
    "zofadra": (ZofadraEngine, bench_zofadra.SIZES, bench_zofadra.zofadra_config, 5),
    "sopanex": (SopanexEngine, bench_sopanex.SIZES, bench_sopanex.sopanex_config, 2),
}
WEIGHT_STD = {"qwen3-4b": 0.006, "qwen3-8b": 0.006, "qwen3.5-4b": 0.02}


def _case(name, model, requests, prompt, new, size="", dtype="bfloat16", ragged=False, portion=0, sample=False):
    return {"name": name, "model": model, "size": size, "dtype": dtype, "requests": requests, "prompt": prompt, "ragged": ragged,
            "portion": portion, "new": new, "sample": sample}


def listed():
    return [
        # a chat turn of one user: a prompt of a line, a short answer; launches and latency
        _case("qwen3-4b-short", "qwen3-4b", 1, 17, 16),
        # the headline benchmark's profile: one request, a page of context, decode after decode
        _case("qwen3-4b-decode", "qwen3-4b", 1, 1024, 64),
        # a document is read and one token asked for: the prompt side of the headline
        _case("qwen3-4b-long-prompt", "qwen3-4b", 1, 10000, 1),
        # a server's batch: many users with prompts of all lengths, answered together
        _case("qwen3-4b-batch", "qwen3-4b", 32, 300, 24, ragged=True),
        # the larger model with top-k / top-p sampling of every step's logits
        _case("qwen3-8b-sampled", "qwen3-8b", 4, 512, 12, sample=True),
        # the hybrid (linear attention beside full attention) with two users
        _case("qwen3.5-4b", "qwen3.5-4b", 2, 1023, 24, ragged=True),
        # latent attention and routed experts, a few users
        _case("duguzen", "duguzen", 4, 901, 16, size="mid", ragged=True),
        # delta rule, matrix memory, routed experts: one user's prompt and answer
        _case("feruzen", "feruzen", 1, 1024, 16, size="mid"),
        # two-map and block-masked attention, channel delta rule; a batch at the small layer sizes
        _case("ramalix", "ramalix", 8, 700, 16, size="small", ragged=True),
        # a long document read in portions, as a scheduler feeds it between other requests
        _case("kukulorn-portions", "kukulorn", 1, 4001, 8, size="mid", portion=1024),
        # single precision, as one checks a checkpoint: no matrix cores, no 16-bit values
        _case("zofadra-float32", "zofadra", 2, 300, 8, size="small", dtype="float32", ragged=True),
        # many users deep in their answers: decoding dominates
        _case("sopanex-decode", "sopanex", 8, 256, 48, size="mid", ragged=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(list(QWEN) + 2 * list(FAMILY))
    case = _case("", model, 1, 1, 1)
    del case["name"]
    case["ragged"] = rng.random() < 0.7
    if model in QWEN:
        case["requests"] = _log_int(rng, 1, 2 if model == "qwen3.5-4b" else 32)
        case["new"] = _log_int(rng, 1, 24)
        total = {"qwen3-4b": 6000, "qwen3-8b": 3000, "qwen3.5-4b": 3000}[model]
        case["sample"] = model != "qwen3.5-4b" and rng.random() < 0.3
    else:
        case["size"] = rng.choice(["small", "mid"])
        case["requests"] = _log_int(rng, 1, 16)
        case["new"] = _log_int(rng, 1, 32)
        total = 4000
        if rng.random() < 0.15:
            case["dtype"], case["size"], total = "float32", "small", 600
    case["prompt"] = _log_int(rng, 5, max(8, total // case["requests"]))
    if model in FAMILY and case["prompt"] > 64 and rng.random() < 0.25:
        case["portion"] = _log_int(rng, 32, case["prompt"])
    return case


# ------------------------------------------------------------------ what a case is made of
def _lengths(case):
    n, p = case["requests"], case["prompt"]
    return [max(1, p - (p * 7 * i) // (8 * n) - 3 * (i % 5)) if case["ragged"] else p for i in range(n)]


def _config(case):
    if case["model"] in QWEN:
        cfg = dict(QWEN[case["model"]])
        if "layer_types" in cfg:
            cfg.update(num_hidden_layers=8, layer_types=cfg["layer_types"][:8])
        return cfg
    _, sizes, make, layers = FAMILY[case["model"]]
    cfg = make(sizes[case["size"]])
    cfg["layers"] = cfg["layers"][:layers]
    if "loop" in cfg:
        cfg["loop"] = dict(cfg["loop"], times=1)
    return cfg


def _tokens(case, seed):
    """(prompts, given continuation [new][requests], random numbers of the sampling [new][requests])"""
    cfg = _config(case)
    rng = np.random.default_rng([seed, 17])
    vocab = cfg.get("vocab") or cfg["vocab_size"]
    prompts = [rng.integers(0, vocab, n).tolist() for n in _lengths(case)]
    given = rng.integers(0, vocab, (case["new"], case["requests"])).tolist()
    return prompts, given, rng.random((case["new"], case["requests"])).tolist()


def _tensors(cfg):
    """[(name, shape, std, mean)] of a family's checkpoint"""
    out = []
    D, V, arch = cfg["width"], cfg["vocab"], cfg["architecture"]

    def lin(name, o, i, gain=1.5):
        out.append((name, (o, i), gain / i ** 0.5, 0.0))

    def vec(name, n, mean=1.0, std=0.2):
        out.append((name, (n,), std, mean))

    def taps(name, rows, k, std=0.4):
        out.append((name, (rows, k), std, 0.0))

    def dyt(name):
        vec(name, D)
        vec(name + ".b", D, 0.0, 0.1)
        out.append((name + ".alpha", (), 0.05, 0.7))

    def glu(p, ff):
        lin(p + ".gate", ff, D)
        lin(p + ".up", ff, D)
        lin(p + ".down", D, ff)

    def moe(p, f, expert, shared_gate=False, router_gain=4.0):
        for e in range(f["router"]["experts"]):
            expert("%s.e%d" % (p, e), f["expert"]["ff"])
        lin(p + ".router", f["router"]["experts"] + f["router"].get("identity", 0), D, router_gain)
        if f.get("shared"):
            expert(p + ".shared", f["shared"]["ff"])
            if shared_gate:
                lin(p + ".shared.sg", 1, D)

    def qkv(q, m, maps=1, v=True):
        lin(q + ".q", m["heads"] * maps * m["dim"], D)
        lin(q + ".k", m["kv_heads"] * maps * m["dim"], D)
        if v:
            lin(q + ".v", m["kv_heads"] * m["vdim"], D)

    def conv_qkv(q, m):
        for n, rows in (("q", m["kv_heads"] * m["dim"]), ("k", m["kv_heads"] * m["dim"]), ("v", m["heads"] * m["vdim"])):
            lin("%s.%s" % (q, n), rows, D)
            taps("%s.%s.conv" % (q, n), rows, m["conv"], 0.5)

    # a tenth where the table is also the head of capped logits: larger ones would all sit at the cap
    out.append(("embed", (V, D), 0.1 if arch == "Kukulorn" else 1.0, 0.0))
    if arch == "Kukulorn":
        lin("loop.in", D, 2 * D, 1.4)
    if arch == "Ramalix":
        taps("loop.step", cfg["loop"]["times"], D, 0.5)
    if arch == "Sopanex":
        taps("bigram", cfg["embedding"]["bigram"]["buckets"] + 1, D, 0.8)
    for i, l in enumerate(cfg["layers"]):
        p, q, m, f = "l%d" % i, "l%d.mix" % i, l["mixer"], l.get("mlp")
        if arch == "Duguzen":
            if "weights_of" in l:
                continue
            for n in (".norm1", ".norm1b", ".norm2", ".norm2b"):
                dyt(p + n)
            lin(q + ".q", m["heads"] * (m["dim"] + m["rot_dim"]), D)
            lin(q + ".dkv", m["kv_rank"] + m["rot_dim"], D)
            vec(q + ".dkv.norm", m["kv_rank"])
            lin(q + ".uk", m["heads"] * m["dim"], m["kv_rank"])
            lin(q + ".uv", m["heads"] * m["vdim"], m["kv_rank"])
            lin(q + ".g", m["heads"], D)
            lin(q + ".o", D, m["heads"] * m["vdim"])
            if f["kind"] == "dense":
                lin(p + ".mlp.up", f["ff"], D)
                lin(p + ".mlp.down", D, f["ff"])
            else:
                moe(p + ".mlp", f, glu)
                vec(p + ".mlp.correction", f["router"]["experts"], 0.0, 0.1)
        elif arch == "Feruzen":
            vec(p + ".norm1", D)
            taps(p + ".canon1", D, cfg["canon"]["taps"])
            vec(p + ".dwa", i + 2, 0.5, 0.2)
            if l["type"] == "delta":
                conv_qkv(q, m)
                lin(q + ".b", m["heads"], D)
                lin(q + ".a", m["heads"], D, 0.5)
                vec(q + ".A_log", m["heads"], -0.5, 0.7)
                vec(q + ".dt_bias", m["heads"], 0.0, 0.5)
                vec(q + ".norm", m["vdim"])
                lin(q + ".g", m["heads"] * m["vdim"], D)
                lin(q + ".o", D, m["heads"] * m["vdim"])
            else:
                a, r = m["left"], m["right"]
                qkv(q + ".left", a)
                vec(q + ".left.q.norm", a["dim"])
                vec(q + ".left.k.norm", a["dim"])
                lin(q + ".left.o", D, a["heads"] * a["vdim"])
                for n, s in (("q", r["dim"]), ("k", r["dim"]), ("v", r["vdim"]), ("g", r["vdim"])):
                    lin("%s.right.%s" % (q, n), r["heads"] * s, D)
                lin(q + ".right.o", D, r["heads"] * r["vdim"])
                vec(q + ".right.norm", r["heads"] * r["vdim"])
                lin(q + ".right.i", r["heads"], D, 0.8)
                vec(q + ".right.i.b", r["heads"], 0.0, 1.0)
                lin(q + ".right.f", r["heads"], D, 0.8)
                vec(q + ".right.f.b", r["heads"], 2.0, 1.0)
            vec(p + ".norm2", D)
            if f["kind"] == "dense":
                glu(p + ".mlp", f["ff"])
            else:
                moe(p + ".mlp", f, glu)
        elif arch == "Ramalix":
            for n in ("1", "2"):
                out.append(("%s.norm%s" % (p, n), (), 0.2, 1.0))
                taps("%s.canon%s" % (p, n), D, cfg["canon"]["taps"])
            if l["type"] == "channel_delta":
                conv_qkv(q, m)
                lin(q + ".b", m["heads"], D)
                lin(q + ".a1", m["a_rank"], D, 1.0)
                lin(q + ".a2", m["heads"] * m["dim"], m["a_rank"], 1.0)
                vec(q + ".A_log", m["heads"], -0.5, 0.7)
                vec(q + ".dt_bias", m["heads"] * m["dim"], 0.0, 0.5)
                vec(q + ".norm", m["vdim"])
                lin(q + ".g1", m["g_rank"], D)
                lin(q + ".g2", m["heads"] * m["vdim"], m["g_rank"])
                lin(q + ".o", D, m["heads"] * m["vdim"])
            else:
                maps = 2 if l["type"] == "attention" else 1
                qkv(q, m, maps)
                lin(q + ".o", D, m["heads"] * m["vdim"])
                if maps == 2:
                    vec(q + ".q.b", m["heads"] * 2 * m["dim"], 0.0, 0.3)
                    vec(q + ".k.b", m["kv_heads"] * 2 * m["dim"], 0.0, 0.3)
                    vec(q + ".v.b", m["kv_heads"] * m["vdim"], 0.0, 0.3)
                    vec(q + ".o.b", D, 0.0, 0.3)
                    for n in ("lq1", "lk1", "lq2", "lk2"):
                        vec("%s.%s" % (q, n), m["dim"], 0.0, 0.4 / m["dim"] ** 0.25)
                else:
                    vec(q + ".sink", m["heads"], 0.5, 1.0)
            moe(p + ".mlp", f, glu, shared_gate=True)
        elif arch == "Kukulorn":
            vec(p + ".norm1", D)
            if l["type"] == "attention":
                a = q
                for n, rows in (("q", m["heads"] * m["dim"]), ("k", m["kv_heads"] * m["dim"]), ("v", m["kv_heads"] * m["vdim"])):
                    taps("%s.%s.conv" % (q, n), rows, m["conv"], 0.5)
                lin(q + ".g", m["heads"] * m["vdim"], D)
                lm = m
            else:
                a, lm, rm = q + ".left", m["left"], m["right"]
                vec(a + ".o.b", D, 0.0, 0.3)
                vec(a + ".q.norm", lm["heads"] * lm["dim"])
                vec(a + ".k.norm", lm["kv_heads"] * lm["dim"])
                taps(a + ".rel", lm["rel_rows"], lm["heads"], 1.0)
                lin(a + ".g", lm["heads"], D)
                inner, gn = rm["heads"] * rm["vdim"], rm["groups"] * rm["state"]
                lin(q + ".right.in", 2 * inner + 2 * gn + rm["heads"], D)
                taps(q + ".right.conv", inner + 2 * gn, rm["conv"], 0.5)
                vec(q + ".right.conv.b", inner + 2 * gn, 0.0, 0.3)
                vec(q + ".right.dt_bias", rm["heads"], -0.5, 0.7)
                vec(q + ".right.A_log", rm["heads"], -0.5, 0.7)
                vec(q + ".right.D", rm["heads"], 1.0, 0.3)
                vec(q + ".right.norm", inner)
                lin(q + ".right.o", D, inner)
                vec(a + ".out", D)
                vec(q + ".right.out", D)
            qkv(a, lm)
            for n, rows in (("q", lm["heads"] * lm["dim"]), ("k", lm["kv_heads"] * lm["dim"]), ("v", lm["kv_heads"] * lm["vdim"])):
                vec("%s.%s.b" % (a, n), rows, 0.0, 0.3)
            lin(a + ".o", D, lm["heads"] * lm["vdim"])
            glu(p + ".mlp", f["ff"])
        elif arch == "Zofadra":
            S, H = cfg["streams"], m["heads"]
            for k in "12":
                vec("%s.norm%s" % (p, k), D)
                vec("%s.hc%s.in" % (p, k), S, 1.0 / S, 0.2)
                vec("%s.hc%s.out" % (p, k), S, 1.0, 0.3)
                out.append(("%s.hc%s.mix" % (p, k), (S, S), 0.2, 0.2))
            if l["type"] == "latent_attention":
                lin(q + ".dq", m["q_rank"], D)
                vec(q + ".dq.norm", m["q_rank"])
                lin(q + ".uq", H * (m["dim"] + m["rot_dim"]), m["q_rank"])
                if "kv_from" not in m:
                    lin(q + ".dkv", m["kv_rank"] + m["rot_dim"], D)
                    vec(q + ".dkv.norm", m["kv_rank"])
                lin(q + ".uk", H * m["dim"], m["kv_rank"])
                lin(q + ".uv", H * m["vdim"], m["kv_rank"])
            elif l["type"] == "attention":
                qkv(q, m)
                vec(q + ".q.norm", H * m["dim"])
                vec(q + ".k.norm", m["kv_heads"] * m["dim"])
            else:
                for n, s in (("q", m["dim"]), ("k", m["dim"]), ("v", m["vdim"]), ("g", m["vdim"])):
                    lin("%s.%s" % (q, n), H * s, D)
                vec(q + ".norm", H * m["vdim"])
            lin(q + ".o", D, H * m["vdim"])
            glu(p + ".mlp", f["ff"])
        else:
            a, r = m["left"], m["right"]
            for n in (".norm1", ".norm1b", ".norm2", ".norm2b"):
                vec(p + n, D, 0.0, 0.2)
            qkv(q + ".left", a, v=False)
            vec(q + ".left.sink", a["heads"], 0.5, 1.0)
            lin(q + ".left.g", a["heads"], D)
            lin(q + ".left.o", D, a["heads"] * a["dim"])
            for n, s in (("q", r["dim"]), ("k", r["dim"]), ("v", r["vdim"]), ("g", r["vdim"])):
                lin("%s.right.%s" % (q, n), r["heads"] * s, D)
            lin(q + ".right.o", D, r["heads"] * r["vdim"])
            vec(q + ".right.norm", r["vdim"])
            lin(q + ".right.a1", r["rank"], D)
            lin(q + ".right.a2", r["heads"] * r["dim"], r["rank"])
            vec(q + ".right.a2.b", r["heads"] * r["dim"], 1.0, 1.5)

            def two(name, ff):
                lin(name + ".up", ff, D)
                lin(name + ".down", D, ff)
            moe(p + ".mlp", f, two, shared_gate=True)
            vec(p + ".mlp.correction", f["router"]["experts"] + f["router"]["identity"], 0.0, 0.02)
    if arch == "Duguzen":
        dyt("final.norm")
    elif arch == "Ramalix":
        out.append(("final.norm", (), 0.1, 1.0))
    else:
        vec("final.norm", D, 0.0 if arch == "Sopanex" else 1.0)
    if arch not in ("Feruzen", "Kukulorn"):
        lin("head", V, D)
    return out


def _checkpoint(case, seed):
    """{name: bf16 tensor on the GPU}, one buffer.  A layer's routed experts share most of their weights, as experts grown from one dense
    layer do, and where there are identity experts a row takes exactly one: a router's near tie that a rounding turns then moves a row
    by little."""
    cfg = _config(case)
    spec = _tensors(cfg)
    counts = [max(1, math.prod(s)) for _, s, _, _ in spec]
    starts = np.cumsum([0] + [(c + 7) // 8 * 8 for c in counts])
    gen = torch.Generator(device="cuda").manual_seed(seed * 7919 + 1)
    flat = torch.randn(int(starts[-1]), device="cuda", dtype=torch.bfloat16, generator=gen)
    out = {}
    for (name, shape, std, mean), n, at in zip(spec, counts, starts):
        t = flat[int(at):int(at) + n]
        t.mul_(std)
        if mean:
            t.add_(mean)
        out[name] = t.view(shape)
        layer, _, expert = name.partition(".mlp.e")
        if expert and not expert.startswith("0."):
            t.mul_(0.03125).add_(out["%s.mlp.e0.%s" % (layer, expert.split(".")[1])].view(-1))
        if case["model"] == "sopanex" and name.endswith(".correction"):
            real = cfg["layers"][0]["mlp"]["router"]["experts"]
            t[real:].fill_(-10.0)
            t[real] = 10.0
    return flat, out


# ------------------------------------------------------------------ the pass
def prepare(case, seed):
    cfg = _config(case)
    prompts, given, uniform = _tokens(case, seed)
    longest, n, new = max(map(len, prompts)), case["requests"], case["new"]
    room = sum((len(p) + new + 15) // 16 + 1 for p in prompts)
    if case["model"] == "qwen3.5-4b":
        eng = Qwen35Engine(cfg, num_kv_pages=room + 8, max_batch_size=n, max_positions=longest + new + 16)
        eng.fill_synthetic(seed=seed, std=WEIGHT_STD[case["model"]])
    elif case["model"] in QWEN:
        eng = Qwen3Engine(cfg, num_kv_pages=room + 8, max_batch_size=8 if n <= 8 else 32, decode_mode=1, max_positions=longest + new + 16)
        eng.fill_synthetic(seed=seed, std=WEIGHT_STD[case["model"]])
    else:
        eng = FAMILY[case["model"]][0](cfg, max_tokens=16 * room, max_requests=n, dtype=case["dtype"])
        flat, tensors = _checkpoint(case, seed)
        host = flat.cpu().view(torch.uint16).numpy()
        base = flat.data_ptr()
        eng.load_tensors({k: host[(t.data_ptr() - base) // 2:][:t.numel()] for k, t in tensors.items()})
        del flat, tensors
    return {"case": case, "engine": eng, "prompts": prompts, "given": given, "uniform": uniform}


def _bf16(bits):
    return torch.from_numpy(bits).view(torch.bfloat16)


def run(state):
    case, eng, prompts, given = state["case"], state["engine"], state["prompts"], state["given"]
    new, out = case["new"], {}
    rids = [eng.new_request() for _ in prompts]
    if case["model"] == "qwen3.5-4b":
        out["prompt_logits"] = np.stack([eng.prefill(r, p, want_logits=True)[1] for r, p in zip(rids, prompts)])
        for s in range(new - 1):
            eng.decode(rids, given[s])
        out["logits"] = eng.decode(rids, given[new - 1], want_logits=True)[1]
    elif case["model"] in QWEN:
        out["prompt_logits"] = _bf16(eng.prefill(rids, prompts, return_logits=True)[1])
        for s in range(new):
            if s == new - 1:
                out["logits"] = _bf16(eng.decode(rids, given[s], return_logits=True)[1])
            else:
                eng.decode(rids, given[s])
            if case["sample"]:
                for c, u in enumerate(state["uniform"][s]):
                    eng.sample(c, 0.8, 50, 0.95, u)
    else:
        portion = case["portion"] or max(map(len, prompts))
        done = [0] * len(prompts)
        ends = {}
        while len(ends) < len(prompts):
            entries, last, row = [], [], 0
            for i, (r, p) in enumerate(zip(rids, prompts)):
                part = p[done[i]:done[i] + portion]
                if part:
                    entries.append((r, part))
                    row += len(part)
                    done[i] += len(part)
                    if done[i] == len(p):
                        last.append((i, row - 1))
            res = eng.step(entries, want=[r for _, r in last], logits=bool(last), tokens=bool(last))
            for (i, _), lg in zip(last, res[0] if last else ()):
                ends[i] = lg
        out["prompt_logits"] = np.stack([ends[i] for i in range(len(prompts))])
        for s in range(new - 1):
            eng.step([(r, [t]) for r, t in zip(rids, given[s])], logits=False, tokens=True)
        out["logits"] = eng.step([(r, [t]) for r, t in zip(rids, given[new - 1])], logits=True, tokens=True)[0]
    for r in rids:
        eng.drop_request(r)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _attention_layers(cfg):
    """[(query heads, flops per (head, query, key), kv values a token leaves, window or None)] of every layer run"""
    out = []
    if "architecture" not in cfg:
        hd = cfg["head_dim"]
        n = cfg["num_hidden_layers"] if "layer_types" not in cfg else sum(t == "full_attention" for t in cfg["layer_types"])
        return [(cfg["num_attention_heads"], 4 * hd, 2 * cfg["num_key_value_heads"] * hd, None)] * n
    for l in cfg["layers"]:
        m = l["mixer"]
        m = m.get("left", m)
        if l["type"] == "latent_attention":
            # keys and values as the heads see them (not through the latent), the latent as what is kept
            kept = 0 if "kv_from" in m else m["kv_rank"] + m["rot_dim"]
            out.append((m["heads"], 2 * (m["dim"] + m["rot_dim"] + m["vdim"]), kept, None))
        elif "kv_heads" in m and l["type"] not in ("delta", "channel_delta"):
            maps = 2 if "diff" in m else 1
            kept = m["dim"] + m["rot"]["dims"] if cfg["architecture"] == "Sopanex" else maps * m["dim"] + m["vdim"]
            window = (m.get("mask") or {}).get("size")
            out.append((m["heads"], 2 * maps * (m["dim"] + m["vdim"]), m["kv_heads"] * kept, window))
    return out


def _state_floats(cfg):
    """values of recurrent state a request holds"""
    if "layer_types" in cfg:
        n = sum(t != "full_attention" for t in cfg["layer_types"])
        return n * cfg["linear_num_value_heads"] * 128 * 128
    total = 0
    for l in cfg.get("layers", ()):
        m = l["mixer"].get("right", l["mixer"])
        if l["type"] in ("delta", "channel_delta", "lightning"):
            total += m["heads"] * m["dim"] * m["vdim"]
        elif "right" in l["mixer"]:
            total += m["heads"] * m["vdim"] * m.get("state", m.get("dim"))
    return total


def _matrices(cfg):
    """(values of the layers' matrices, of all routed experts' matrices, of the head's; share of the experts that a row takes)"""
    if "architecture" not in cfg:
        H, I, V, hd = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"], cfg["head_dim"]
        qd, kvd, L = cfg["num_attention_heads"] * hd, cfg["num_key_value_heads"] * hd, cfg["num_hidden_layers"]
        if "layer_types" not in cfg:
            return L * (2 * qd * H + 2 * kvd * H + 3 * I * H), 0, V * H, 0.0
        full = sum(t == "full_attention" for t in cfg["layer_types"])
        kd, vd, vh = 128 * cfg["linear_num_key_heads"], 128 * cfg["linear_num_value_heads"], cfg["linear_num_value_heads"]
        lin = (2 * kd + vd) * H + 2 * vd * H + 2 * vh * H
        return full * (3 * qd + 2 * kvd) * H + (L - full) * lin + 3 * L * I * H, 0, V * H, 0.0
    dense = experts = 0
    walks = {}
    for i, l in enumerate(cfg["layers"]):
        walks[l.get("weights_of", i)] = walks.get(l.get("weights_of", i), 0) + 1
    for name, shape, _, _ in _tensors(cfg):
        if len(shape) != 2 or name in ("embed", "bigram", "head"):
            continue
        times = walks.get(int(name[1:].split(".")[0]), 1) if name[0] == "l" and name[1].isdigit() else 1
        if ".mlp.e" in name:
            experts += times * math.prod(shape)
        else:
            dense += times * math.prod(shape)
    routers = [l["mlp"]["router"] for l in cfg["layers"] if l.get("mlp", {}).get("kind") == "moe"]
    share = (routers[0]["top"] - (1 if routers[0].get("identity") else 0)) / routers[0]["experts"] if routers else 0.0
    return dense, experts, cfg["vocab"] * cfg["width"], share


def work(case):
    """Every call (the prompts' step or steps, every decode step) reads the weights it needs once - the experts that its rows choose, for
    routed layers -, the keys and values behind its rows once per request and the recurrent state once each way."""
    cfg, lens = _config(case), _lengths(case)
    size = 4 if case["dtype"] == "float32" else 2
    dense, experts, head, share = _matrices(cfg)
    att, state = _attention_layers(cfg), _state_floats(cfg)
    portion = case["portion"] or max(lens)
    steps = [[(min(portion, n - at), at) for n in lens if n > at] for at in range(0, max(lens), portion)]
    if case["model"] == "qwen3.5-4b":
        steps = [[(n, 0)] for n in lens]
    steps += [[(1, n + s) for n in lens] for s in range(case["new"])]
    nbytes = flops = 0.0
    for k, entries in enumerate(steps):
        rows = sum(r for r, _ in entries)
        ends = len(entries)
        nbytes += size * (dense + head + experts * (1.0 - (1.0 - share) ** rows if experts else 0.0)) + 8.0 * state * ends
        flops += 2.0 * rows * (dense + experts * share) + 2.0 * ends * head + 6.0 * state * rows
        for heads, per, kept, window in att:
            for r, at in entries:
                pairs = r * at + r * (r + 1) // 2
                if window:
                    pairs = min(pairs, r * window)
                nbytes += size * kept * (min(at + r, window + r) if window else at + r)
                flops += heads * per * pairs
    return {"bytes": nbytes, "flops": flops}


# four times the error of the logits against `exact`, the largest of the listed cases and of a hundred drawn ones, and no more than three
# hundredths: values in bf16 along 36 layers (8 hybrid ones) or 2 .. 5 layers; a router's near tie that a rounding turns moves a whole row
# (duguzen, ramalix, sopanex)
REL = {"qwen3-4b": 0.03, "qwen3-8b": 0.03, "qwen3.5-4b": 0.03, "duguzen": 0.03, "feruzen": 0.026, "ramalix": 0.03, "kukulorn": 0.03,
       "zofadra": 0.03, "sopanex": 0.03}


def tolerance(case):
    return {"rel": 2e-5 if case["dtype"] == "float32" else REL[case["model"]]}


# ------------------------------------------------------------------ the same numbers in 64 bits, plain torch
def _synthetic(index, seed, std, mean, single=False):
    """the numbers a seeded Qwen engine gives the weights at these positions: a hash of the position, two uniform numbers of 24 bits, one
    normal number in single precision"""
    def shr(z, k):
        return (z >> k) & ((1 << (64 - k)) - 1)

    def wrap(c):
        return c - (1 << 64) if c >= 1 << 63 else c
    z = index * wrap(0x9E3779B97F4A7C15) + seed
    z = (z ^ shr(z, 30)) * wrap(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * wrap(0x94D049BB133111EB)
    z = z ^ shr(z, 31)
    u1 = (shr(z, 40).float() + 1.0) * (1.0 / 16777217.0)
    u2 = (shr(z, 16) & 0xFFFFFF).float() * (1.0 / 16777216.0)
    v = mean + std * (torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(6.2831853 * u2))
    return v if single else v.bfloat16()


class _SyntheticWeights:
    """tensors of a seeded Qwen engine, drawn in the engine's order"""

    def __init__(self, seed, std):
        self.base, self.count, self.std = seed * 1000003, 0, std

    def next(self, rows, cols=1, std=None, mean=0.0, single=False):
        self.count += 1
        std = self.std if std is None else std
        return functools.partial(self._values, self.base + self.count, rows, cols, std, mean, single)

    @staticmethod
    def _values(seed, rows, cols, std, mean, single, pick=None):
        """all rows, or the picked ones, in double precision"""
        pick = torch.arange(rows, device="cuda") if pick is None else pick
        out = torch.empty(len(pick), cols, dtype=F64, device="cuda")
        step = max(1, (1 << 26) // cols)
        for lo in range(0, len(pick), step):
            index = pick[lo:lo + step, None] * cols + torch.arange(cols, device="cuda")
            out[lo:lo + step] = _synthetic(index, seed, std, mean, single)
        return out if cols > 1 else out[:, 0]


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _frequencies(dims, base):
    return [base ** (-2.0 * i / dims) for i in range(dims // 2)]


def _turn(x, freqs, neighbours, amplitude=1.0):
    """x [n, heads, d]: pairs of the first 2 len(freqs) values turn by position times frequency"""
    n, dims = x.shape[0], 2 * len(freqs)
    ang = torch.arange(n, dtype=F64, device=x.device)[:, None] * torch.tensor(freqs, dtype=F64, device=x.device)
    c, s = amplitude * torch.cos(ang)[:, None], amplitude * torch.sin(ang)[:, None]
    if neighbours:
        u, v = x[..., 0:dims:2], x[..., 1:dims:2]
        r = torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
    else:
        u, v = x[..., :dims // 2], x[..., dims // 2:dims]
        r = torch.cat([u * c - v * s, v * c + u * s], -1)
    return torch.cat([r, x[..., dims:]], -1)


def _attend(q, k, v, scale, see=None, change=None, sink=None):
    """q [n, H, d], k [n, G, d], v [n, G, dv] -> [n, H, dv]; see(i, j) narrows the causal keys, change(scores, head, distance) alters scores"""
    n, H = q.shape[:2]
    G = k.shape[1]
    out = q.new_empty(n, H, v.shape[2])
    at = torch.arange(n, device=q.device)
    for lo in range(0, n, 2048):
        hi = min(n, lo + 2048)
        i, j = at[lo:hi, None], at[None, :hi]
        ok = j <= i
        if see is not None:
            ok = ok & see(i, j)
        for h in range(H):
            g = h // (H // G)
            s = (q[lo:hi, h] @ k[:hi, g].T) * scale
            if change is not None:
                s = change(s, h, i - j)
            s = s.masked_fill(~ok, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(hi - lo, 1)], 1)
            out[lo:hi, h] = torch.softmax(s, -1)[:, :hi] @ v[:hi, g]
    return out


def _conv(x, taps, bias=None):
    """causal convolution per channel, the last tap on the current token"""
    k = taps.shape[1]
    pad = torch.cat([x.new_zeros(k - 1, x.shape[1]), x])
    out = sum(pad[j:j + len(x)] * taps[:, j] for j in range(k))
    return out if bias is None else out + bias


def _recur(q, k, v, decay, beta=None):
    """q, k [n, H, d], v [n, H, dv], decay [n, H, d or 1], beta [n, H]: S <- diag(decay) S; with beta the delta rule, else S += k v^T; S^T q"""
    n, H, d = q.shape
    S = q.new_zeros(H, d, v.shape[2])
    out = q.new_empty(n, H, v.shape[2])
    for t in range(n):
        S = decay[t][:, :, None] * S
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None]
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out


def _spread(x, heads):
    return x.repeat_interleave(heads // x.shape[1], 1)


def _exact_qwen3(cfg, seed, std, seqs):
    H, I, L, V, hd = (cfg[k] for k in ("hidden_size", "intermediate_size", "num_hidden_layers", "vocab_size", "head_dim"))
    Hq, G, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    w = _SyntheticWeights(seed, std)
    embed = w.next(V, H)
    head = embed if cfg["tie_word_embeddings"] else w.next(V, H)
    final = w.next(H, std=0.1, mean=1.0)()
    freqs = _frequencies(hd, cfg["rope_theta"])
    lens = [len(s) for s in seqs]
    x = embed(pick=torch.tensor([t for s in seqs for t in s], device="cuda"))
    for _ in range(L):
        qkv, o = w.next((Hq + 2 * G) * hd, H), w.next(H, Hq * hd)
        qn, kn = w.next(hd, std=0.1, mean=1.0)(), w.next(hd, std=0.1, mean=1.0)()
        gate_up, down = w.next(2 * I, H), w.next(H, I)
        ln1, ln2 = w.next(H, std=0.1, mean=1.0)(), w.next(H, std=0.1, mean=1.0)()
        a = (_rms(x, eps) * ln1) @ qkv().T
        parts = []
        for b in a.split(lens):
            q, k, v = b.view(len(b), -1, hd).split([Hq, G, G], 1)
            q, k = _turn(_rms(q, eps) * qn, freqs, False), _turn(_rms(k, eps) * kn, freqs, False)
            parts.append(_attend(q, k, v, hd ** -0.5).flatten(1))
        x = x + torch.cat(parts) @ o().T
        g, u = ((_rms(x, eps) * ln2) @ gate_up().T).chunk(2, -1)
        x = x + (Fn.silu(g) * u) @ down().T
    return (_rms(x, eps) * final).split(lens), lambda rows: rows @ head().T


def _exact_qwen35(cfg, seed, std, seqs):
    H, I, V, hd = (cfg[k] for k in ("hidden_size", "intermediate_size", "vocab_size", "head_dim"))
    Hq, G, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    kh, vh, taps = cfg["linear_num_key_heads"], cfg["linear_num_value_heads"], cfg["linear_conv_kernel_dim"]
    C, Z = (2 * kh + vh) * 128, vh * 128
    w = _SyntheticWeights(seed, std)
    embed = w.next(V, H)
    final = w.next(H, std=0.1)()
    freqs = _frequencies(int(hd * cfg["partial_rotary_factor"]), cfg["rope_theta"])
    lens = [len(s) for s in seqs]
    x = embed(pick=torch.tensor([t for s in seqs for t in s], device="cuda"))
    for kind in cfg["layer_types"]:
        ln1, ln2 = w.next(H, std=0.1)(), w.next(H, std=0.1)()
        gate, up, down = w.next(I, H), w.next(I, H), w.next(H, I)
        h = _rms(x, eps) * (1.0 + ln1)
        parts = []
        if kind == "full_attention":
            wq, wk, wv, wo = w.next(2 * Hq * hd, H), w.next(G * hd, H), w.next(G * hd, H), w.next(H, Hq * hd)
            qn, kn = w.next(hd, std=0.1)(), w.next(hd, std=0.1)()
            for q, k, v in zip(*((h @ m().T).split(lens) for m in (wq, wk, wv))):
                q = q.view(len(q), Hq, 2, hd)
                q, g = q[:, :, 0], q[:, :, 1]
                k, v = k.view(len(k), G, hd), v.view(len(v), G, hd)
                q, k = _turn(_rms(q, eps) * (1.0 + qn), freqs, False), _turn(_rms(k, eps) * (1.0 + kn), freqs, False)
                parts.append((_attend(q, k, v, hd ** -0.5) * torch.sigmoid(g)).flatten(1))
        else:
            wqkv, wz, wb, wa = w.next(C, H), w.next(Z, H), w.next(vh, H), w.next(vh, H)
            conv, dt, wo = w.next(C, taps, std=0.3)(), w.next(vh, std=0.5)(), w.next(H, Z)
            rate, norm = torch.exp(w.next(vh, std=0.5, single=True)()), w.next(128, std=0.1, mean=1.0, single=True)()
            for a, z, b, s in zip(*((h @ m().T).split(lens) for m in (wqkv, wz, wb, wa))):
                q, k, v = Fn.silu(_conv(a, conv)).view(len(a), -1, 128).split([kh, kh, vh], 1)
                q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-12) for t in (q, k))
                decay = torch.exp(-rate * Fn.softplus(s + dt))[..., None]
                y = _recur(_spread(q, vh) * 128 ** -0.5, _spread(k, vh), v, decay, torch.sigmoid(b))
                parts.append((_rms(y, eps) * norm).flatten(1) * Fn.silu(z))
        x = x + torch.cat(parts) @ wo().T
        h = _rms(x, eps) * (1.0 + ln2)
        x = x + (Fn.silu(h @ gate().T) * (h @ up().T)) @ down().T
    return (_rms(x, eps) * (1.0 + final)).split(lens), lambda rows: rows @ embed().T


class _Named:
    """w[name] in double precision; lin(x, name) = x W^T"""

    def __init__(self, tensors):
        self.t = tensors

    def __getitem__(self, name):
        return self.t[name].to(F64)

    def lin(self, x, name):
        return x @ self[name].T


def _routed(w, p, h, idx, val, experts, expert):
    out = torch.zeros_like(h)
    for e in range(experts):
        rows, col = torch.nonzero(idx == e, as_tuple=True)
        if len(rows):
            out.index_add_(0, rows, val[rows, col][:, None] * expert(h[rows], "%s.e%d" % (p, e)))
    return out


def _exact_duguzen(cfg, w, toks):
    eps = cfg["norm"]["eps"]

    def dyt(x, n):
        return torch.tanh(w[n + ".alpha"] * x) * w[n] + w[n + ".b"]
    x = w["embed"][toks]
    n = len(toks)
    for i, l in enumerate(cfg["layers"]):
        m, f, p = l["mixer"], l["mlp"], "l%d" % l.get("weights_of", i)
        q = p + ".mix"
        h = dyt(x, p + ".norm1")
        d, dr, r = m["dim"], m["rot_dim"], m["kv_rank"]
        freqs = _frequencies(m["rot"]["dims"], m["rot"]["base"])
        qq = w.lin(h, q + ".q").view(n, m["heads"], d + dr)
        a = w.lin(h, q + ".dkv")
        c = _rms(a[:, :r], eps) * w[q + ".dkv.norm"]
        kr = _turn(a[:, None, r:], freqs, False).expand(n, m["heads"], dr)
        qq = torch.cat([qq[..., :d], _turn(qq[..., d:], freqs, False)], -1)
        k = torch.cat([w.lin(c, q + ".uk").view(n, m["heads"], d), kr], -1)
        v = w.lin(c, q + ".uv").view(n, m["heads"], m["vdim"])
        y = _attend(qq, k, v, m["scale"]) * torch.sigmoid(w.lin(h, q + ".g"))[..., None]
        x = x + dyt(w.lin(y.flatten(1), q + ".o"), p + ".norm1b")
        h = dyt(x, p + ".norm2")
        p += ".mlp"
        if f["kind"] == "dense":
            y = w.lin(torch.relu(w.lin(h, p + ".up")) ** 2, p + ".down")
        else:
            rt = f["router"]
            s = torch.sigmoid(w.lin(h, p + ".router"))
            G, E = rt["groups"]["count"], rt["experts"]
            choice = (s + w[p + ".correction"]).view(n, G, E // G)
            kept = choice.topk(2, -1).values.sum(-1).topk(rt["groups"]["keep"], -1).indices
            ok = torch.zeros(n, G, dtype=torch.bool, device=x.device).scatter_(1, kept, True)
            idx = choice.masked_fill(~ok[..., None], -math.inf).flatten(1).topk(rt["top"], -1).indices
            y = _routed(w, p, h, idx, s.gather(1, idx), E,
                        lambda t, e: w.lin(Fn.silu(w.lin(t, e + ".gate")) * w.lin(t, e + ".up"), e + ".down"))
        x = x + dyt(y, p[:-4] + ".norm2b")
    return dyt(x, "final.norm"), "head"


def _exact_feruzen(cfg, w, toks):
    eps, parts = cfg["norm"]["eps"], cfg["norm"]["groups"]
    n = len(toks)

    def grms(y, name):
        return _rms(y.view(n, parts, -1), eps).flatten(1) * w[name]

    def glu(t, p, limit):
        g, u = torch.clamp(w.lin(t, p + ".gate"), max=limit), torch.clamp(w.lin(t, p + ".up"), -limit, limit)
        return w.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + ".down")
    x = w["embed"][toks]
    stack = [x]
    for i, l in enumerate(cfg["layers"]):
        p, q, m, f = "l%d" % i, "l%d.mix" % i, l["mixer"], l["mlp"]
        h = x + _conv(x, w[p + ".canon1"])
        if l["type"] == "delta":
            H = m["heads"]
            qq, k, v = (Fn.silu(_conv(w.lin(h, q + s), w[q + s + ".conv"])).view(n, -1, m[z])
                        for s, z in ((".q", "dim"), (".k", "dim"), (".v", "vdim")))
            qq, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (qq, k))
            decay = torch.exp(-torch.exp(w[q + ".A_log"]) * Fn.softplus(w.lin(h, q + ".a") + w[q + ".dt_bias"]))
            o = _recur(_spread(qq, H) * m["dim"] ** -0.5, _spread(k, H), v, decay[..., None], torch.sigmoid(w.lin(h, q + ".b")))
            y = w.lin((_rms(o, eps) * w[q + ".norm"]).flatten(1) * Fn.silu(w.lin(h, q + ".g")), q + ".o")
        else:
            a, r, ql, qr = m["left"], m["right"], q + ".left", q + ".right"
            freqs = _frequencies(a["rot"]["dims"], a["rot"]["base"])
            qq, k, v = (w.lin(h, ql + s).view(n, -1, a[z]) for s, z in ((".q", "dim"), (".k", "dim"), (".v", "vdim")))
            qq, k = (_turn(_rms(t, eps) * w[ql + s], freqs, True) for t, s in ((qq, ".q.norm"), (k, ".k.norm")))
            y = m["left_scale"] * w.lin(_attend(qq, k, v, a["scale"]).flatten(1), ql + ".o")
            H, d, dv, cap = r["heads"], r["dim"], r["vdim"], r["gate_cap"]
            qq = w.lin(h, qr + ".q").view(n, H, d) * d ** -0.5
            k, v = w.lin(h, qr + ".k").view(n, H, d), w.lin(h, qr + ".v").view(n, H, dv)
            ig, fg = (cap * torch.tanh((w.lin(h, qr + s) + w[qr + s + ".b"]) / cap) for s in (".i", ".f"))
            fg = Fn.logsigmoid(fg)
            S, nv, mm = x.new_zeros(H, d, dv), x.new_zeros(H, d), x.new_zeros(H)
            o = x.new_empty(n, H, dv)
            for t in range(n):
                top = torch.maximum(fg[t] + mm, ig[t])
                keep, put = torch.exp(fg[t] + mm - top)[:, None], torch.exp(ig[t] - top)[:, None]
                kk = put * k[t]
                S = keep[..., None] * S + kk[..., None] * v[t][:, None]
                nv, mm = keep * nv + kk, top
                den = torch.maximum((nv * qq[t]).sum(-1).abs(), torch.exp(-mm)) + 1e-6
                o[t] = torch.bmm(qq[t][:, None], S)[:, 0] / den[:, None]
            o = _rms(o, eps).flatten(1) * w[qr + ".norm"] * torch.sigmoid(w.lin(h, qr + ".g"))
            y = y + m["right_scale"] * w.lin(o, qr + ".o")
        x = x + grms(y, p + ".norm1")
        if f["kind"] == "dense":
            y = glu(x, p + ".mlp", f["limit"])
        else:
            val, idx = torch.softmax(w.lin(x, p + ".mlp.router"), -1).topk(f["router"]["top"], -1)
            y = _routed(w, p + ".mlp", x, idx, val, f["router"]["experts"], lambda t, e: glu(t, e, f["expert"]["limit"]))
            y = y + glu(x, p + ".mlp.shared", f["shared"]["limit"])
        stack.append(x + grms(y, p + ".norm2"))
        x = sum(c * s for c, s in zip(w[p + ".dwa"], stack))
    return grms(x, "final.norm"), "embed"


def _exact_ramalix(cfg, w, toks):
    eps, mult, n = cfg["norm"]["eps"], cfg["residual_mult"], len(toks)

    def swiglu(t, p):
        return w.lin(Fn.silu(w.lin(t, p + ".gate")) * w.lin(t, p + ".up"), p + ".down")
    x = w["embed"][toks] + w["loop.step"][0]
    at = torch.arange(n, device=x.device)
    for i, l in enumerate(cfg["layers"]):
        p, q, m, f = "l%d" % i, "l%d.mix" % i, l["mixer"], l["mlp"]
        h = _rms(x, eps) * w[p + ".norm1"]
        h = h + _conv(h, w[p + ".canon1"])
        if l["type"] == "channel_delta":
            H, d = m["heads"], m["dim"]
            qq, k, v = (Fn.silu(_conv(w.lin(h, q + s), w[q + s + ".conv"])).view(n, -1, m[z])
                        for s, z in ((".q", "dim"), (".k", "dim"), (".v", "vdim")))
            qq, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (qq, k))
            a = w.lin(w.lin(h, q + ".a1"), q + ".a2") + w[q + ".dt_bias"]
            decay = torch.exp(-torch.exp(w[q + ".A_log"])[:, None] * Fn.softplus(a).view(n, H, d))
            o = _recur(_spread(qq, H) * d ** -0.5, _spread(k, H), v, decay, torch.sigmoid(w.lin(h, q + ".b")))
            gate = torch.sigmoid(w.lin(w.lin(h, q + ".g1"), q + ".g2"))
            y = w.lin((_rms(o, eps) * w[q + ".norm"]).flatten(1) * gate, q + ".o")
        elif l["type"] == "attention":
            H, G, d = m["heads"], m["kv_heads"], m["dim"]
            qq, k = ((w.lin(h, q + s) + w[q + s + ".b"]).view(n, c, 2, d) for s, c in ((".q", H), (".k", G)))
            v = (w.lin(h, q + ".v") + w[q + ".v.b"]).view(n, G, m["vdim"])
            t = m["q_temp"]
            qq = qq * (1.0 + t["coef"] * torch.log(torch.div(at + 1, t["every"], rounding_mode="floor").to(F64) + 1.0))[:, None, None, None]
            lam = torch.exp((w[q + ".lq1"] * w[q + ".lk1"]).sum()) - torch.exp((w[q + ".lq2"] * w[q + ".lk2"]).sum()) + m["diff"]
            o1, o2 = (_attend(qq[:, :, c], k[:, :, c], v, m["scale"]) for c in range(2))
            y = w.lin((_rms(o1 - lam * o2, eps) * (1.0 - m["diff"])).flatten(1), q + ".o") + w[q + ".o.b"]
        else:
            freqs, block = _frequencies(m["rot"]["dims"], m["rot"]["base"]), m["mask"]["size"]
            qq, k, v = (w.lin(h, q + s).view(n, -1, m[z]) for s, z in ((".q", "dim"), (".k", "dim"), (".v", "vdim")))
            qq, k = _turn(qq, freqs, True), _turn(k, freqs, True)
            o = _attend(qq, k, v, m["scale"], see=lambda a, b: torch.div(a, block, rounding_mode="floor") ==
                        torch.div(b, block, rounding_mode="floor"), sink=w[q + ".sink"])
            y = w.lin(o.flatten(1), q + ".o")
        x = x + mult * y
        h = _rms(x, eps) * w[p + ".norm2"]
        h = h + _conv(h, w[p + ".canon2"])
        p, r = p + ".mlp", f["router"]
        s = torch.softmax(w.lin(h, p + ".router"), -1).view(n, r["groups"]["count"], -1)
        kept = s.max(-1).values.topk(r["groups"]["keep"], -1).indices
        ok = torch.zeros(s.shape[:2], dtype=torch.bool, device=x.device).scatter_(1, kept, True)
        val, idx = s.masked_fill(~ok[..., None], -1.0).flatten(1).topk(r["top"], -1)
        y = _routed(w, p, h, idx, val / (val.sum(-1, keepdim=True) + 1e-20), r["experts"], swiglu)
        x = x + mult * (y + swiglu(h, p + ".shared") * torch.sigmoid(w.lin(h, p + ".shared.sg")))
    return _rms(x, eps) * w["final.norm"] * cfg["logit_scale"], "head"


def _exact_kukulorn(cfg, w, toks):
    eps, n = cfg["norm"]["eps"], len(toks)
    x0 = w["embed"][toks]
    x = w.lin(torch.cat([x0, x0], -1), "loop.in")
    for i, l in enumerate(cfg["layers"]):
        p, q, m = "l%d" % i, "l%d.mix" % i, l["mixer"]
        h = _rms(x, eps) * w[p + ".norm1"]
        if l["type"] == "attention":
            qq, k, v = (_conv(w.lin(h, q + s) + w[q + s + ".b"], w[q + s + ".conv"]).view(n, -1, 128) for s in (".q", ".k", ".v"))
            rot = m["rot"]
            sc, freqs = rot["scaling"], []
            for fr in _frequencies(rot["dims"], rot["base"]):
                turns = sc["original"] * fr / (2.0 * math.pi)
                s = min(1.0, max(0.0, (turns - sc["low"]) / (sc["high"] - sc["low"])))
                freqs.append((1.0 - s) * fr / sc["factor"] + s * fr)
            qq, k = (_rms(_turn(t, freqs, False), eps) for t in (qq, k))
            cap = m["softcap"]
            o = _attend(qq, k, v, m["scale"], change=lambda s, head, dist: cap * torch.tanh(s / cap)).flatten(1)
            y = w.lin(o * torch.sigmoid(w.lin(h, q + ".g")), q + ".o")
        else:
            a, r, ql, qr = m["left"], m["right"], q + ".left", q + ".right"
            qq, k = ((_rms(w.lin(h, ql + s) + w[ql + s + ".b"], eps) * w[ql + s + ".norm"]).view(n, -1, 128) for s in (".q", ".k"))
            v = (w.lin(h, ql + ".v") + w[ql + ".v.b"]).view(n, -1, 128)
            rel = w[ql + ".rel"]
            B, far, mask = rel.shape[0], a["bias_max"], a["mask"]
            hb = B // 2
            dist = torch.arange(n, dtype=F64, device=x.device)
            steps = torch.floor(torch.log(torch.clamp(dist, min=1.0) / hb) / math.log(far / hb) * (B - hb))
            rows = rel[torch.where(dist < hb, dist, torch.clamp(hb + steps, max=B - 1)).long()]
            o = _attend(qq, k, v, a["scale"], see=lambda i_, j_: (i_ - j_ < mask["size"]) | (j_ < mask["keep_first"]),
                        change=lambda s, head, d_: s + rows[:, head][d_.clamp(min=0)])
            left = w.lin((o * torch.sigmoid(w.lin(h, ql + ".g"))[..., None]).flatten(1), ql + ".o") + w[ql + ".o.b"]
            H, P, N, G = r["heads"], r["vdim"], r["state"], r["groups"]
            z, xbc, dt = w.lin(h, qr + ".in").split([H * P, H * P + 2 * G * N, H], -1)
            xx, Bm, Cm = Fn.silu(_conv(xbc, w[qr + ".conv"], w[qr + ".conv.b"])).split([H * P, G * N, G * N], -1)
            xx, Bm, Cm = xx.reshape(n, H, P), _spread(Bm.reshape(n, G, N), H), _spread(Cm.reshape(n, G, N), H)
            dt = Fn.softplus(dt + w[qr + ".dt_bias"])
            y = _recur(Cm, Bm * dt[..., None], xx, torch.exp(-torch.exp(w[qr + ".A_log"]) * dt)[..., None])
            y = (y + w[qr + ".D"][:, None] * xx).flatten(1) * Fn.silu(z)
            right = w.lin(_rms(y.view(n, r["norm_groups"], -1), eps).flatten(1) * w[qr + ".norm"], qr + ".o")
            y = 0.5 * (_rms(left, eps) * w[ql + ".out"] + _rms(right, eps) * w[qr + ".out"])
        p += ".mlp"
        x = x + y + w.lin(torch.relu(w.lin(h, p + ".gate")) * w.lin(h, p + ".up"), p + ".down")
    return _rms(x, eps) * w["final.norm"], "embed"


def _exact_zofadra(cfg, w, toks):
    eps, mult, n = cfg["norm"]["eps"], cfg["residual_mult"], len(toks)

    def norm(x, name):
        d = x - x.mean(-1, keepdim=True)
        return _rms(d, eps) * w[name]

    def join(X, p, y):
        return torch.einsum("snd,st->tnd", X, w[p + ".mix"]) + mult * w[p + ".out"][:, None, None] * y
    X = (w["embed"][toks] * cfg["embedding"]["scale"])[None].repeat(cfg["streams"], 1, 1)
    latents = {}
    for i, l in enumerate(cfg["layers"]):
        p, q, m = "l%d" % i, "l%d.mix" % i, l["mixer"]
        H = m["heads"]
        h = norm((w[p + ".hc1.in"][:, None, None] * X).sum(0), p + ".norm1")
        if l["type"] == "latent_attention":
            d, r = m["dim"], m["kv_rank"]
            freqs = _frequencies(m["rot"]["dims"], m["rot"]["base"])
            if "kv_from" not in m:
                a = w.lin(h, q + ".dkv")
                latents[i] = _rms(a[:, :r], eps) * w[q + ".dkv.norm"], _turn(a[:, None, r:], freqs, True)
            c, kr = latents[m.get("kv_from", i)]
            qq = w.lin(_rms(w.lin(h, q + ".dq"), eps) * w[q + ".dq.norm"], q + ".uq").view(n, H, -1)
            qq = torch.cat([qq[..., :d], _turn(qq[..., d:], freqs, True)], -1)
            k = torch.cat([w.lin(c, q + ".uk").view(n, H, d), kr.expand(n, H, m["rot_dim"])], -1)
            o = _attend(qq, k, w.lin(c, q + ".uv").view(n, H, m["vdim"]), m["scale"]).flatten(1)
        elif l["type"] == "attention":
            qq, k = ((_rms(w.lin(h, q + s), eps) * w[q + s + ".norm"]).view(n, -1, m["dim"]) for s in (".q", ".k"))
            size = m["mask"]["size"]
            o = _attend(qq, k, w.lin(h, q + ".v").view(n, -1, m["vdim"]), m["scale"], see=lambda a, b: a - b < size,
                        change=lambda s, head, dist: s - 2.0 ** (-8.0 * (head + 1) / H) * dist).flatten(1)
        else:
            qq, k, v = (Fn.silu(w.lin(h, q + s)).view(n, H, -1) for s in (".q", ".k", ".v"))
            decay = torch.tensor(m["decay"], dtype=F64, device=X.device)[None, :, None].expand(n, H, 1)
            o = _rms(_recur(qq, k, v, decay).flatten(1), eps) * w[q + ".norm"] * torch.sigmoid(w.lin(h, q + ".g"))
        X = join(X, p + ".hc1", w.lin(o, q + ".o"))
        h = norm((w[p + ".hc2.in"][:, None, None] * X).sum(0), p + ".norm2")
        g = Fn.gelu(w.lin(h, p + ".mlp.gate"), approximate="tanh")
        X = join(X, p + ".hc2", w.lin(g * w.lin(h, p + ".mlp.up"), p + ".mlp.down"))
    return norm(X.sum(0), "final.norm"), "head"


def _exact_sopanex(cfg, w, toks):
    eps, n, bg = cfg["norm"]["eps"], len(toks), cfg["embedding"]["bigram"]

    def zrms(x, name):
        return _rms(x, eps) * (1.0 + w[name])

    def expert(t, p):
        return w.lin(Fn.gelu(w.lin(t, p + ".up")), p + ".down")
    rows = torch.cat([toks.new_tensor([bg["buckets"]]), (toks[:-1] * bg["mul_prev"] + toks[1:] * bg["mul_cur"]) % bg["buckets"]])
    x = w["embed"][toks] * cfg["embedding"]["scale"] + w["bigram"][rows]
    for i, l in enumerate(cfg["layers"]):
        p, m, f = "l%d" % i, l["mixer"], l["mlp"]
        a, r, ql, qr = m["left"], m["right"], p + ".mix.left", p + ".mix.right"
        h = zrms(x, p + ".norm1")
        sc, dims, base = a["rot"]["scaling"], a["rot"]["dims"], a["rot"]["base"]
        lo, hi = (dims * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base)) for t in (sc["fast"], sc["slow"]))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
        freqs = []
        for j, fr in enumerate(_frequencies(dims, base)):
            ramp = min(max((j - lo) / max(hi - lo, 0.001), 0.0), 1.0)
            freqs.append(fr / sc["factor"] * ramp + fr * (1.0 - ramp))
        amp = 0.1 * math.log(sc["factor"]) + 1.0
        qq, v = w.lin(h, ql + ".q").view(n, -1, a["dim"]), w.lin(h, ql + ".k").view(n, -1, a["dim"])
        o = _attend(_turn(qq, freqs, False, amp), _turn(v, freqs, False, amp), v, a["scale"], sink=w[ql + ".sink"])
        y = m["left_scale"] * w.lin((o * torch.sigmoid(w.lin(h, ql + ".g"))[..., None]).flatten(1), ql + ".o")
        H, d = r["heads"], r["dim"]
        qq, k, v = (w.lin(h, qr + s).view(n, H, -1) for s in (".q", ".k", ".v"))
        z = w.lin(w.lin(h, qr + ".a1"), qr + ".a2") + w[qr + ".a2.b"]
        o = _recur(qq * d ** -0.5, k, v, torch.exp(Fn.logsigmoid(z) / r["tau"]).view(n, H, d))
        o = (_rms(o, eps) * w[qr + ".norm"]).flatten(1) * Fn.silu(w.lin(h, qr + ".g"))
        x = x + zrms(y + m["right_scale"] * w.lin(o, qr + ".o"), p + ".norm1b")
        h = zrms(x, p + ".norm2")
        q, rt = p + ".mlp", f["router"]
        s = torch.softmax(w.lin(h, q + ".router"), -1)
        idx = (s + w[q + ".correction"]).topk(rt["top"], -1).indices
        val = s.gather(1, idx)
        val = val / (val.sum(-1, keepdim=True) + 1e-20) * rt["scale"]
        y = _routed(w, q, h, idx, val, rt["experts"], expert) + (val * (idx >= rt["experts"])).sum(-1, keepdim=True) * h
        y = y + expert(h, q + ".shared") * torch.sigmoid(w.lin(h, q + ".shared.sg"))
        x = x + zrms(y, p + ".norm2b")
    return zrms(x, "final.norm"), "head"


EXACT = {"duguzen": _exact_duguzen, "feruzen": _exact_feruzen, "ramalix": _exact_ramalix, "kukulorn": _exact_kukulorn,
         "zofadra": _exact_zofadra, "sopanex": _exact_sopanex}


def exact(case, seed):
    cfg = _config(case)
    prompts, given, _ = _tokens(case, seed)
    seqs = [p + [row[i] for row in given] for i, p in enumerate(prompts)]
    if case["model"] in QWEN:
        rows, head = (_exact_qwen35 if case["model"] == "qwen3.5-4b" else _exact_qwen3)(cfg, seed, WEIGHT_STD[case["model"]], seqs)
    else:
        flat, tensors = _checkpoint(case, seed)
        w = _Named(tensors)
        done = [EXACT[case["model"]](cfg, w, torch.tensor(s, device="cuda")) for s in seqs]
        rows = [r for r, _ in done]
        cap = cfg.get("logit_softcap")

        def head(r):
            lg = w.lin(r, done[0][1])
            return cap * torch.tanh(lg / cap) if cap else lg
    # rows that were asked for: the end of the prompt and the last continued token
    at_prompt = head(torch.stack([r[len(p) - 1] for r, p in zip(rows, prompts)]))
    at_end = head(torch.stack([r[-1] for r in rows]))
    return {"prompt_logits": at_prompt.cpu().numpy(), "logits": at_end.cpu().numpy()}
