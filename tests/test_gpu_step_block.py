"""The block of a step's metadata on its way to the device: the kernel that fetches it at the head of a captured step, and engines whose block outgrows its
first 4096 words between replays."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

WORDS = 4096      # requested whatever the count is


@pytest.mark.parametrize("count", [0, 1, 3, 4, 5, 4095, 4096, 4097, 8191, 8192, 8193, 20000])
def test_fetched_words_are_the_counted_ones(count):
    """up to the count rounded up to four words, and none behind them; the count is read when the launch runs"""
    from pegainfer_amd import ops_blocks as B
    room = max(WORDS, (count + 3) // 4 * 4)
    src = torch.empty(4 + room, dtype=torch.int32, pin_memory=True)
    src.copy_(torch.arange(1000, 1004 + room, dtype=torch.int32))
    dst = torch.full((room + 64,), -7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert src.data_ptr() % 16 == 0
    src[0] = count
    assert B.ffi.lib().pegainfer_fetch_words(dst.data_ptr(), src[4:].data_ptr(), src.data_ptr(), B._stream()) == 0
    got, n = dst.cpu(), (count + 3) // 4 * 4
    assert torch.equal(got[:n], src[4:4 + n]) and bool((got[n:] == -7).all())


@pytest.mark.parametrize("family", ["duguzen", "feruzen", "kukulorn", "ramalix", "sopanex", "zofadra"])
def test_replayed_steps_whose_block_outgrows_its_first_words(family):
    """24 requests, then 640 (more than 4096 words), then 24 again, several steps each: the same bits as steps that are never captured"""
    C = importlib.import_module(family + "_common")
    cfg = C.config_tiny()
    w = C.weights_for(cfg, 5, "bfloat16") if hasattr(C, "weights_for") else C.random_weights(cfg, 5)
    out = []
    for eager in (False, True):
        eng = C.engine_for(cfg, w, "bfloat16", max_tokens=16 * 1400, max_requests=640)
        eng.debug_hidden_enable(eager)
        r, got = [eng.new_request() for _ in range(640)], []
        for some in (r[:24], r[24:332], r[332:]):
            eng.step([(q, [(3 * q + k) % cfg["vocab"] for k in range(1 + q % 3)]) for q in some], want=[])
        for step, use in enumerate([r[:24]] * 3 + [r] * 3 + [r[:24]] * 2 + [r] * 14):      # most contexts take a second page at the end
            lg, tk = eng.step([(q, [(q + 7 * step) % cfg["vocab"]]) for q in use], want=list(range(0, len(use), 5)), tokens=True)
            got += [lg, tk]
        out.append(got)
        eng.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out)) and len(out[0]) == len(out[1])
