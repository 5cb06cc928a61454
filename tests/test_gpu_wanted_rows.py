"""Steps whose wanted rows are all of them in order (the last layer's closing launch norms them for the output table), against the same
steps with the rows asked for in another order or in part (a launch of their own picks and norms them): same logits, row by row.  Decode steps and prompts."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MODELS = [("ramalix", "a"), ("ramalix", "only_delta"), ("duguzen", "a"), ("kukulorn", "a"), ("sopanex", "a"), ("zofadra", "a")]


def _tolerance(dtype):
    """the layers' bits are the same; the last norm's sum may be ordered otherwise, which moves a normed value by a rounding of its type (2^-24, 2^-9)
    and a logit, a sum of such terms, by less than four of them against the largest"""
    return 2.0 ** -17 if dtype == "float32" else 2.0 ** -7


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("model,name", MODELS)
def test_all_rows_in_order_and_picked_rows_agree(model, name, dtype):
    C = importlib.import_module(model + "_common")
    cfg = C.config_for(name, dtype) if hasattr(C, "config_for") else getattr(C, "config_" + name)()
    w = C.weights_for(cfg, 5, dtype) if hasattr(C, "weights_for") else C.random_weights(cfg, 5)
    toks = C.tokens_for(cfg, 40, 3)
    n = 3

    def run(want):
        eng = C.engine_for(cfg, w, dtype)
        reqs = [eng.new_request() for _ in range(n)]
        eng.step([(r, toks[: 5 + 3 * i]) for i, r in enumerate(reqs)])
        out = [eng.step([(r, [toks[20 + 4 * t + i]]) for i, r in enumerate(reqs)], want=want) for t in range(4)]
        eng.close()
        return out

    every, tol = run(None), _tolerance(dtype)
    for want in ([2, 1, 0], [1], [0, 1, 2]):
        for a, b in zip(every, run(want)):
            assert np.abs(a[want] - b).max() <= tol * np.abs(a).max(), (want, float(np.abs(a[want] - b).max()))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("model,name", MODELS)
def test_prompts_that_want_every_row(model, name, dtype):
    C = importlib.import_module(model + "_common")
    cfg = C.config_for(name, dtype) if hasattr(C, "config_for") else getattr(C, "config_" + name)()
    w = C.weights_for(cfg, 5, dtype) if hasattr(C, "weights_for") else C.random_weights(cfg, 5)
    toks, rows = C.tokens_for(cfg, 40, 3), 33

    def run(want):
        eng = C.engine_for(cfg, w, dtype)
        reqs = [eng.new_request() for _ in range(3)]
        out = eng.step([(reqs[0], toks[:20]), (reqs[1], toks[20:32]), (reqs[2], toks[32:33])], want=want)
        eng.close()
        return out
    every = run(list(range(rows)))
    assert every.shape[0] == rows
    for want in (list(range(rows))[::-1], [0, 19, 31, 32], list(range(rows - 1))):
        assert np.abs(every[want] - run(want)).max() <= _tolerance(dtype) * np.abs(every).max(), want
