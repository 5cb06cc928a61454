"""Requests of a step whose values are no numbers beside requests that are sound: the sound ones' logits are bit for bit what they are beside
sound companions.  A row that is no number has no eligible expert, so all its choices fall on expert 0, which then has more pairs than
the step has rows."""
import numpy as np
import pytest
import torch

import duguzen_common
import feruzen_common
import ramalix_common
import sopanex_common

pytestmark = pytest.mark.gpu

FAMILIES = {"duguzen": duguzen_common, "feruzen": feruzen_common, "ramalix": ramalix_common, "sopanex": sopanex_common}


@pytest.mark.parametrize("rows,bad", [(2, 1), (4, 2), (8, 5), (16, 10), (17, 11)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("family", FAMILIES)
def test_rows_of_no_number_leave_their_companions_alone(family, dtype, rows, bad):
    C = FAMILIES[family]
    cfg = C.config_b()
    w = C.weights_for(cfg, 5, dtype) if hasattr(C, "weights_for") else C.random_weights(cfg, 5)
    w["embed"] = w["embed"].clone()
    w["embed"][3] = float("nan")
    toks = [4 + (7 * i) % 60 for i in range(rows)]
    runs = []
    for companions in ([3] * bad, toks[:bad]):
        eng = C.engine_for(cfg, w, dtype, max_requests=rows)
        ids = [eng.new_request() for _ in range(rows)]
        got = eng.step([(r, [t]) for r, t in zip(ids, companions + toks[bad:])], want=list(range(rows)))
        runs.append(np.array(got[bad:], dtype=np.float32))
        eng.close()
    assert np.isfinite(np.delete(runs[1], 3, axis=1)).all()
    assert np.array_equal(runs[0].view(np.uint32), runs[1].view(np.uint32))


@pytest.mark.parametrize("per_tile", [1, 3, 16])
def test_tables_of_few_rows_hold_no_tile_past_their_cut(per_tile):
    """an expert with more pairs than a tile takes is cut, every position lies in one tile; other cuts between the two kinds are refused"""
    from pegainfer_amd import ops_blocks as B
    expert = torch.tensor([[0, 0, 0, 0], [0, 1, 2, 4], [4, 0, 1, 2], [0, 0, 0, 0]], dtype=torch.int32)
    pos_pair, pos_row, tg, t0, tr, nt, max_tiles = B.route_sort(expert.cuda(), 5, rows_per_tile=per_tile)
    seen = []
    for t in range(int(nt)):
        g, r0, n = int(tg[t]), int(t0[t]), int(tr[t])
        assert 0 < n <= per_tile and all(int(expert.view(-1)[int(pos_pair[p])]) == g for p in range(r0, r0 + n))
        seen += list(range(r0, r0 + n))
    assert seen == list(range(16)) and sorted(pos_pair.tolist()) == list(range(16))
    for refused in (17, 63, 65, 127):
        with pytest.raises(Exception):
            B.route_sort(expert.cuda(), 5, rows_per_tile=refused)
