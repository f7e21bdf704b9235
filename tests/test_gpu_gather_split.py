"""Gathers through source regions (2^24 elements and more) against torch's own
indexing, bit for bit: element widths, ragged last tiles (one element, one short
of a tile), sources smaller and larger than the index vector, repeated indexes,
indexes in order (gathered directly) and all in one region, dst in place of the
indexes, another stream, and capture in a graph."""
from __future__ import annotations

import pytest
from gpu_util import say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N = 1 << 24
DTYPE = {1: torch.uint8, 2: torch.int16, 4: torch.int32, 8: torch.int64}


def _indexes(pattern: str, n: int, nsrc: int) -> torch.Tensor:
    gen = torch.Generator(device="cuda").manual_seed(n)
    if pattern == "order":
        return torch.arange(n, device="cuda") % nsrc
    if pattern == "far":  # neighbours far apart, yet each tile in few regions
        i = torch.arange(n, device="cuda")
        return (i % 2) * (nsrc // 2) + (i // 2) % (nsrc // 2)
    return torch.randint(0, nsrc, (n,), generator=gen, device="cuda")


def _source(width: int, n: int) -> torch.Tensor:
    gen = torch.Generator(device="cuda").manual_seed(width)
    return torch.randint(-128 if width > 1 else 0, 127, (n,), generator=gen, device="cuda").to(DTYPE[width])


@pytest.mark.parametrize("width", [1, 2, 4, 8])
@pytest.mark.parametrize("pattern,n,nsrc", [("random", N, N), ("random", N + 1, 5 * N // 2), ("random", N + 16383, 777),
                                            ("random", 2 * N + 3, N // 2 + 5), ("order", N + 5, N), ("far", N + 77, N)])
def test_gather_equals_indexing(handle, width, pattern, n, nsrc):
    src, idx = _source(width, nsrc), _indexes(pattern, n, nsrc)
    dst = torch.zeros(n, dtype=src.dtype, device="cuda")
    say(f"gather {pattern} n={n} nsrc={nsrc} width={width}")
    handle.gather(src, idx, dst)
    assert torch.equal(dst, src[idx])


def test_gather_over_its_indexes(handle):
    src, idx = _source(8, N), _indexes("random", N + 9, N)
    want = src[idx]
    say("gather over its indexes")
    handle.gather(src, idx, idx)
    assert torch.equal(idx, want)


@pytest.mark.parametrize("width,times", [(1, 40), (2, 24), (4, 15), (4, 25), (8, 7), (8, 13)])
def test_gather_from_a_sparse_source(handle, width, times):
    """Sources far larger than the index vector, on both sides of where the split
    gives way to a direct gather."""
    n = N + 11
    src, idx = _source(width, times * n), _indexes("random", n, times * n)
    dst = torch.zeros(n, dtype=src.dtype, device="cuda")
    say(f"gather from {times} times as many elements, width={width}")
    handle.gather(src, idx, dst)
    assert torch.equal(dst, src[idx])


def _best_ms(call) -> float:
    call()
    ms = []
    for _ in range(5):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        for _ in range(5):
            call()
        t1.record()
        torch.cuda.synchronize()
        ms.append(t0.elapsed_time(t1) / 5)
    return min(ms)


def test_gather_from_a_sparse_source_costs_no_more(handle):
    """Where hardly two indexes share a line the call takes what a direct gather (a
    captured call) does, not the split's passes on top (a quarter more)."""
    src, idx = _source(8, 64 * N), _indexes("random", N, 64 * N)
    dst = torch.zeros(N, dtype=torch.int64, device="cuda")
    handle.gather(src, idx, dst)
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    try:
        with torch.cuda.graph(graph, stream=stream):
            handle.set_stream(torch.cuda.current_stream().cuda_stream)
            handle.gather(src, idx, dst)
    finally:
        handle.set_stream(0)
    say("time of a sparse gather")
    direct, call = _best_ms(graph.replay), _best_ms(lambda: handle.gather(src, idx, dst))
    print(direct, call)
    assert call < 1.12 * direct


@pytest.mark.parametrize("every", [1, 3, 100, N])
def test_gather_of_indexes_past_32_bits(handle, every):
    """One index in `every` lies past 2^32: such an element is gathered again after
    its tile was put in place; most of them, and all is gathered directly."""
    n = N + 5
    src = torch.zeros((1 << 32) + n, dtype=torch.uint8, device="cuda")
    src[:n] = _source(1, n)
    src[1 << 32:] = _source(1, n) + 101
    idx = _indexes("random", n, n)
    idx[::every] += 1 << 32
    dst = torch.zeros(n, dtype=torch.uint8, device="cuda")
    say(f"gather, one index in {every} past 2^32")
    handle.gather(src, idx, dst)
    assert torch.equal(dst, src[idx])


def test_gather_over_its_indexes_past_32_bits(handle):
    """dst over idx: a tile with such an index is left to the last kernel."""
    n = N + 5
    src = torch.empty((1 << 32) + n, dtype=torch.int64, device="cuda")
    src[:n] = _source(8, n)
    src[1 << 32:] = _source(8, n) * 3
    idx = _indexes("random", n, n)
    idx[::50_000] += 1 << 32
    want = src[idx]
    say("gather over its indexes, some past 2^32")
    handle.gather(src, idx, idx)
    assert torch.equal(idx, want)


def test_few_indexes_past_32_bits_cost_no_multiple(handle):
    """One index in a hundred past 2^32 leaves no tile of 16,384 without one: such a
    gather took 2.2 times as long as one without."""
    n = 2 * N
    src = torch.zeros((1 << 32) + n, dtype=torch.uint8, device="cuda")
    idx, dst = _indexes("random", n, n), torch.zeros(n, dtype=torch.uint8, device="cuda")
    say("time of a gather with indexes past 2^32")
    ms = [_best_ms(lambda: handle.gather(src, idx, dst))]
    idx[::100] += 1 << 32
    ms.append(_best_ms(lambda: handle.gather(src, idx, dst)))
    print(ms)
    assert ms[1] < 1.7 * ms[0]


def test_gather_on_changing_streams(handle):
    """Two streams in turn: the scratch of one call is not written by the next
    before it is read."""
    src = [_source(4, N + i) for i in range(6)]
    idx = [_indexes("random", N + 3 * i, N + i) for i in range(6)]
    dst = [torch.zeros(N + 3 * i, dtype=torch.int32, device="cuda") for i in range(6)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    say("gathers on two streams")
    try:
        for i in range(6):
            handle.set_stream(streams[i % 2].cuda_stream)
            handle.gather(src[i], idx[i], dst[i])
        torch.cuda.synchronize()
    finally:
        handle.set_stream(0)
    for i in range(6):
        assert torch.equal(dst[i], src[i][idx[i]]), i


def test_gather_in_a_graph(handle):
    """Captured, the call takes the direct kernel: no scratch is kept by the graph."""
    src, idx = _source(4, N), _indexes("random", N, N)
    dst = torch.zeros(N, dtype=torch.int32, device="cuda")
    handle.gather(src, idx, dst)
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    say("gather in a graph")
    try:
        with torch.cuda.graph(graph, stream=stream):
            handle.set_stream(torch.cuda.current_stream().cuda_stream)
            handle.gather(src, idx, dst)
    finally:
        handle.set_stream(0)
    for seed in range(3):
        src.copy_(_source(4, N) + seed)
        dst.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dst, src[idx]), seed
        handle.gather(src, _indexes("random", N + seed, N), torch.empty(N + seed, dtype=torch.int32, device="cuda"))
