"""A sampled token comes back through a word that the draw writes itself: call after call, beside decode steps, each gets its own, and a call that has no
place for the token is refused."""
import ctypes
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_tokens_of_calls_in_a_row():
    from oracle.bf16 import bf16_from_bits
    from pegainfer_amd.qwen3 import Qwen3Engine
    golden = os.path.join(os.path.dirname(__file__), "golden")
    meta = json.load(open(os.path.join(golden, "qwen3_tiny_golden.json")))
    eng = Qwen3Engine(meta["config"], num_kv_pages=64, max_batch_size=2).load_safetensors(os.path.join(golden, "qwen3_tiny.safetensors"))
    rids = [eng.new_request(), eng.new_request()]
    _, logits = eng.prefill(rids, [meta["cases"][2]["prompt_tokens"], meta["cases"][1]["prompt_tokens"]], return_logits=True)
    for step in range(4):
        best = [int(np.argmax(bf16_from_bits(row))) for row in logits]
        # one kept token is the largest logit's, whichever form draws it
        for _ in range(3):
            assert [eng.sample(c, 0.7, 1, 0.9, 0.3) for c in (0, 1)] == best
            assert [eng.sample(c, 0.0, 0, 1.0, 0.3) for c in (1, 0)] == best[::-1]
        _, logits = eng.decode(rids, best, return_logits=True)
    assert eng.lib.pegainfer_qwen3_sample(eng.h, 0, ctypes.c_float(0.7), 1, ctypes.c_float(0.9), ctypes.c_float(0.3), None) != 0
    assert eng.sample(0, 0.7, 1, 0.9, 0.3) == int(np.argmax(bf16_from_bits(logits[0])))
