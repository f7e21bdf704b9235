"""Rank sorts whose samples fill the pinned buffer: keys and payloads of the
samples are read back together, in blocks that only just fit it, so splitters,
bucket sizes and the result must equal the oracle's re-run whatever the buffer
held before."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from gpu_util import assert_bits_equal, dev, host, say
from gpusort_amd import HYKSORT, HYPERQUICKSORT, SAMPLESORT, GpusortError

pytestmark = pytest.mark.gpu

CASES = [  # algorithm, ranks, keys a rank, samples a rank, key and payload types
    ("samplesort", 1024, 5 * 1024 + 3, 8, np.uint32, np.uint32),
    ("samplesort", 660, 5 * 660 + 1, 8, np.float64, np.uint32),
    ("samplesort", 600, 5 * 600 + 2, 8, np.uint64, np.int64),
    ("samplesort", 520, 5 * 520 + 9, 8, np.int64, np.uint64),
    ("hyperquicksort", 16, 40_000, 20_000, np.uint64, np.int64),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-p{c[1]}-{np.dtype(c[4]).name}-{np.dtype(c[5]).name}")
def test_samples_that_fill_the_buffer(handle, case):
    algo, p, per, s, kdt, vdt = case
    r = np.random.RandomState(p)
    off = np.arange(p + 1, dtype=np.uint64) * np.uint64(per)
    n = int(off[-1])
    keys = r.randint(0, 1 << 62, n, dtype=np.int64)
    keys = (keys % 1_000_003).astype(kdt) if kdt is np.float64 else keys.view(np.uint64).astype(kdt)
    vals = r.permutation(n).astype(vdt)
    want_k, want_v, want = oracle.vrank(keys, off.astype(np.int64), vals, algorithm=algo, k_way=8, samples_per_rank=s)
    for turn in range(2):  # from two fill levels of the buffer
        tk, tv = dev(keys), dev(vals)
        say(f"rank reads {algo} p={p} n={n} turn={turn}")
        got = handle.vrank_sort(tk, off, tv, algorithm={"samplesort": SAMPLESORT, "hyperquicksort": HYPERQUICKSORT}[algo],
                                k_way=8, samples_per_rank=s)
        assert_bits_equal(got["splitters"], want["splitters"], "splitters")
        assert np.array_equal(got["bucket_sizes"].astype(np.int64), want["bucket_sizes"]), "bucket sizes"
        assert np.array_equal(got["final_rank_sizes"].astype(np.int64), want["final_rank_sizes"])
        assert_bits_equal(host(tk), want_k, "keys")
        assert_bits_equal(host(tv), want_v, "payloads")


def test_a_call_that_fails_has_waited_for_its_stream(handle):
    """An error in the middle of a rank sort (more samples than the selection
    takes) leaves nothing queued that still reads the buffer."""
    torch = pytest.importorskip("torch")
    off = np.array([0, 30_000, 60_000], dtype=np.uint64)
    keys = np.random.RandomState(3).randint(0, 1 << 31, 60_000).astype(np.uint32)
    stream, other = torch.cuda.Stream(), torch.cuda.Stream()
    tk = dev(keys)
    torch.cuda.synchronize()
    try:
        handle.set_stream(stream)
        with torch.cuda.stream(stream):
            torch.cuda._sleep(20_000_000)
        say("rank sort with too many samples")
        with pytest.raises(GpusortError, match="exceeds"):
            handle.vrank_sort(tk, off, algorithm=HYKSORT, k_way=2, samples_per_rank=1 << 24)
        assert stream.query(), "the failed call left work queued"
        handle.set_stream(other)
        tk = dev(keys)
        torch.cuda.synchronize()
        handle.vrank_sort(tk, off, algorithm=HYKSORT, k_way=2, samples_per_rank=32)
    finally:
        handle.set_stream(0)
    assert_bits_equal(host(tk), np.sort(keys), "keys")
