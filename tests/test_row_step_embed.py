"""A step's first row read from the embedding table (pegainfer_row_step_embed): the row that the table's own launch leaves, and what the entry refuses."""
import ctypes

import pytest
import torch

ROWS, D = 5, 1028


def _call(B, dt, embed, ids, stream=0, **parts):
    from pegainfer_amd import ffi
    p = lambda v: v.data_ptr() if torch.is_tensor(v) else v  # noqa: E731
    q = B.RowStepDesc(d=D, rows=ROWS, dtype={torch.bfloat16: 0, torch.float32: 1}[dt], **{k: p(v) for k, v in parts.items()})
    return ffi.lib().pegainfer_row_step_embed(ctypes.c_void_p(ctypes.addressof(q)), ctypes.c_void_p(p(embed)), ctypes.c_void_p(p(ids)), ctypes.c_void_p(stream))


@pytest.mark.skipif(torch.cuda.is_available(), reason="addresses stand for device memory: on the host, where no launch can follow")
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_refusals(built_libs, dt):
    """no table, no ids, another source of rows, the forms that have none from a table, and a table off its alignment: refused before a launch"""
    import pegainfer_amd.ops_blocks as B
    at, table = 1 << 20, 1 << 21                        # never read: every call is refused by its arguments
    form = dict(x_out=at, gain=at, eps=1e-5, n_out=at)
    off = 4 if dt == torch.bfloat16 else 8
    for embed, ids, parts in [(None, at, {}), (table, None, {}), (table, at, dict(x_in=at)), (table, at, dict(row_index=at)),
                              (table, at, dict(y_pairs=at, weight=at, top=1)), (table, at, dict(groups=4, y=at, n_out=None)), (table + off, at, {}),
                              (table, at, dict(x_out=at + 8)), (table, at, dict(n_out=at + 4)), (table, at, dict(bias=at))]:
        assert _call(B, dt, embed, ids, **dict(form, **parts)) == 1, (embed, ids, parts)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_rows_of_the_table(dt):
    """the sum alone, with the added vector, and with norm and convolution: the bits of the table's own launch in front of pegainfer_row_step"""
    import pegainfer_amd.ops_blocks as B
    g = torch.Generator().manual_seed(5)
    draw = lambda *s, t=dt: torch.randn(*s, generator=g).to(t).cuda()  # noqa: E731
    V, stride = 77, 3 * D + 4
    embed, vec, one, cw = draw(V, D), draw(D), draw(1), draw(D, 4)
    ids = torch.tensor([76, 0, 3, 3, 41], dtype=torch.int32).cuda()
    slots = torch.tensor([4, 0, 2, 1, 3], dtype=torch.int32).cuda()
    x = B.embed_f32(embed, ids)
    stream = torch.cuda.current_stream().cuda_stream
    for parts in (dict(), dict(add_vec=vec), dict(gain=one, eps=1e-5), dict(add_vec=vec, gain=one, eps=1e-5)):
        got, want = torch.full_like(x, 9), x.clone()
        outs = []
        for src in (got, want):
            state, conv = torch.ones(5, stride, device="cuda"), torch.zeros(ROWS, D, dtype=dt, device="cuda")
            cv = dict(conv_w=cw, conv_state=state, conv_slot_stride=stride, conv_slot=slots, conv_out=conv) if "gain" in parts else {}
            if src is got:
                assert _call(B, dt, embed, ids, stream, x_out=got, **parts, **cv) == 0
            else:
                B.row_step(dt, ROWS, D, x_in=want, x_out=want, **parts, **cv)
            outs.append((src, state, conv))
        for a, b in zip(*outs):
            assert torch.equal(a, b), list(parts)
