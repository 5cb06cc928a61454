"""Times of products that stand beside each other: what differs between the two of a pair is worth a few per cent, and a form that has lost its way out or its
order of loads is a quarter slower or more.  The line lies between what was measured of both; a form is slower every time, so the best of three counts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ratio(first, second, n, limit):
    """median time of `first` over that of `second`, in turn; the best of three"""
    best = float("inf")
    for f in (first, second):
        for i in range(n):
            f(i)
    for _ in range(3):
        times = ([], [])
        for _ in range(7):
            for k, f in enumerate((first, second)):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in "ab")
                a.record()
                for i in range(n):
                    f(i)
                b.record()
                b.synchronize()
                times[k].append(a.elapsed_time(b))
        best = min(best, sorted(times[0])[3] / sorted(times[1])[3])
        if best < limit:
            break
    return best


# 4 mod 8 against whole chunks: 1.0 where halves of a chunk leave in 8 bytes, 1.6 / 2.3 / 3.3 value by value
@pytest.mark.parametrize("cut,whole,T,K", [((4100, 1020, 1024), (4096, 1024, 1024), 2048, 2560), ((8192, 1028, 1020), (8192, 1024, 1024), 2100, 1024),
                                           ((4096, 2052, 2044), (4096, 2048, 2048), 4096, 256)])
def test_segments_inside_a_chunk_cost_what_whole_ones_cost(cut, whole, T, K):
    from pegainfer_amd import ops as P
    W, X = torch.randn(sum(cut), K, device="cuda").bfloat16(), torch.randn(T, K, device="cuda").bfloat16()
    ys = [[torch.empty(T, m, device="cuda", dtype=torch.bfloat16) for m in parts] for parts in (cut, whole)]
    assert _ratio(lambda i: P.gemm_split3_into(W, X, *ys[0]), lambda i: P.gemm_split3_into(W, X, *ys[1]), 10, 1.3) < 1.3


# few rows with their norm in front against the product alone: 1.11 / 1.21 / 1.19 / 1.14 where the norm waits for its rows, 1.34 / 1.33 / 1.36 / 1.26 where it
# waits for the weights behind them too
@pytest.mark.parametrize("T,K,residual,limit", [(4, 1024, True, 1.24), (9, 2560, False, 1.27), (9, 3072, False, 1.28), (3, 3072, False, 1.20)])
def test_norm_in_front_of_few_rows_does_not_wait_for_weights(T, K, residual, limit):
    from pegainfer_amd import ffi
    M, lib, s = 6144, ffi.lib(), torch.cuda.current_stream().cuda_stream
    n = int(4e8 / (2 * M * K))                       # more weights than the last cache holds
    W = torch.randn(n, M, K, device="cuda").bfloat16()
    X, R, left, gain = (torch.randn(T, K, device="cuda").bfloat16() for _ in range(4))
    Y = torch.empty(T, M, device="cuda", dtype=torch.bfloat16)
    w, x, y, plain = [v.data_ptr() for v in W], X.data_ptr(), Y.data_ptr(), (None, None, None)
    normed = (R.data_ptr() if residual else None, gain.data_ptr(), left.data_ptr() if residual else None)

    def run(i, before):
        assert lib.pegainfer_gemv_fused(w[i], x, y, M, T, K, *before, 1e-6, 0, s) == 0
    assert _ratio(lambda i: run(i, normed), lambda i: run(i, plain), n, limit) < limit


# 32 columns (tiles of 32) against 33 (of 64): 0.92 with a ring of weights that is requested at once, 1.04 / 1.05 with one of 14 tiles
@pytest.mark.parametrize("M", [16384, 12292])
def test_32_columns_take_no_longer_than_33(M):
    from pegainfer_amd import ffi
    K, lib, s = 1024, ffi.lib(), torch.cuda.current_stream().cuda_stream
    W, X = torch.randn(int(4e8 / (2 * M * K)), M, K, device="cuda").bfloat16(), torch.randn(33, K, device="cuda").bfloat16()
    Y = torch.empty(33, M, device="cuda", dtype=torch.bfloat16)
    w, x, y = [v.data_ptr() for v in W], X.data_ptr(), Y.data_ptr()
    assert _ratio(lambda i: lib.gemm_cuda(w[i], x, y, M, 32, K, s), lambda i: lib.gemm_cuda(w[i], x, y, M, 33, K, s), len(w), 0.98) < 0.98


def test_ten_rounds_of_tiles_beside_a_held_unit():
    """One wave of another stream keeps the 256 x 256 tiles off its compute unit: 1.1 of the time alone where a workgroup takes a tile, 1.4 and more where
    workgroups stay for the whole launch and the one that found no unit begins as the others are through."""
    import time
    from pegainfer_amd import ffi, ops
    M, T, K, lib = 19456, 8192, 512, ffi.lib()
    W, X = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(T, K, device="cuda").bfloat16()
    Y = torch.empty(T, M, device="cuda", dtype=torch.bfloat16)
    here, there = torch.cuda.Stream(), torch.cuda.Stream()

    def timed(stream, f):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in "ab")
        with torch.cuda.stream(stream):
            a.record()
            f()
            b.record()
        b.synchronize()
        return a.elapsed_time(b)
    ops.gemm_into(W, X, Y)
    torch.cuda.synchronize()
    gemm = lambda: lib.gemm_cuda(W.data_ptr(), X.data_ptr(), Y.data_ptr(), M, T, K, here.cuda_stream)  # noqa: E731
    torch.cuda._sleep(1000)
    cycles = 1000000 / timed(there, lambda: torch.cuda._sleep(1000000))      # a millisecond
    alone, beside = sorted(timed(here, gemm) for _ in range(9))[4], []
    for _ in range(20):
        with torch.cuda.stream(there):
            torch.cuda._sleep(int(cycles * (4 * alone + 3)))
        time.sleep(0.001)
        took = timed(here, gemm)
        if not there.query():                          # the unit was held all the time
            beside.append(took)
        there.synchronize()
        if len(beside) == 5:
            break
    assert beside
    assert sorted(beside)[len(beside) // 2] / alone < 1.25


# one tile of tokens against two: 0.65 where the weights, which have one reader, are loaded past the caches, 0.78 where they push each other out
def test_weights_of_a_single_tile_of_tokens_pass_the_caches():
    from pegainfer_amd import ffi
    M, K, lib, s = 65536, 4096, ffi.lib(), torch.cuda.current_stream().cuda_stream
    W, X = torch.randn(2, M, K, device="cuda").bfloat16(), torch.randn(257, K, device="cuda").bfloat16()
    Y = torch.empty(257, M, device="cuda", dtype=torch.bfloat16)
    w, x, y = [v.data_ptr() for v in W], X.data_ptr(), Y.data_ptr()
    assert _ratio(lambda i: lib.gemm_cuda(w[i % 2], x, y, M, 256, K, s), lambda i: lib.gemm_cuda(w[i % 2], x, y, M, 257, K, s), 6, 0.71) < 0.71
