"""64-bit keys in many small clusters (composite keys: the upper half one of many
ids): runs of a few to some hundred keys that agree in the digits sorted by, of every
length around the words, the rounds and the longest run that one workgroup compares,
across its chunks, among random keys and with no other key, and a cost that is no
multiple of other keys'."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu

_SIZES = [2, 3, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 254, 255, 256, 257, 258, 300, 511, 513, 1000]


def _clusters(sizes, r, low_bits: int) -> np.ndarray:
    ids = r.permutation(1 << 22)[: len(sizes)].astype(np.uint64) * np.uint64(1021)
    x = np.repeat(ids << np.uint64(32), sizes)
    return x + r.randint(0, 1 << low_bits, x.size, dtype=np.uint64)


def _keys(name: str, n: int, seed: int) -> np.ndarray:
    r = np.random.RandomState(seed)
    if name == "some":  # one key in a hundred, in runs of all sizes; low digits of few values, so with equal keys
        c = _clusters(_SIZES * max(1, n // 100 // sum(_SIZES)), r, 7)
    elif name == "mixed":  # every key, in runs of 1 to 80
        sizes = r.randint(1, 81, n // 40)
        c = _clusters(sizes[np.cumsum(sizes) <= n], r, 32)
    else:  # ordered but for a few keys
        sizes = r.randint(1, 81, n // 40)
        c = np.sort(_clusters(sizes[np.cumsum(sizes) <= n], r, 32))
        at = r.choice(c.size - 1, 50, replace=False)
        c[at], c[at + 1] = c[at + 1], c[at]
    x = r.randint(0, 1 << 63, n, dtype=np.uint64) * np.uint64(2)
    x[: c.size] = c
    return x if name == "nearly" else x[r.permutation(n)]


@pytest.mark.parametrize("vdt", [None, np.uint32, np.uint64], ids=lambda t: "none" if t is None else np.dtype(t).name)
@pytest.mark.parametrize("name,n", [("some", 600_011), ("some", (1 << 22) + 2047), ("some", (1 << 23) + 2049),
                                    ("mixed", 40_001), ("mixed", (1 << 22) + 1), ("mixed", (1 << 24) + 255),
                                    ("nearly", 3_000_017)])
def test_runs_within_a_chunk(handle, name, n, vdt):
    keys = _keys(name, n, n)
    for kdt, desc in ((np.uint64, False), (np.int64, True)):
        k = keys.view(kdt)
        vals = None if vdt is None else np.arange(n).astype(vdt)
        order = stable_order(k, desc)
        say(f"clusters {name} {np.dtype(kdt).name} n={n} vals={vdt} desc={desc}")
        tk, tv = dev(k), None if vals is None else dev(vals)
        if vals is None:
            handle.sort_keys(tk, descending=desc)
        else:
            handle.sort_pairs(tk, tv, descending=desc)
            assert_bits_equal(host(tv), vals[order], f"{name} payloads")
        assert_bits_equal(host(tk), k[order], f"{name} keys")


@pytest.mark.parametrize("vdt", [None, np.uint32], ids=["none", "uint32"])
def test_runs_at_the_ends_of_segments(handle, vdt):
    """The same keys in every segment, so that runs of one touch equal digits of the next."""
    parts = [_keys("some", 600_011, 1), _keys("mixed", 40_000, 2), _keys("mixed", 40_000, 2), np.zeros(0, np.uint64),
             _keys("mixed", 500_009, 3), _keys("nearly", 100_003, 4)]
    parts += [np.sort(_keys("mixed", 20_011, 5))[::-1][:s].copy() for s in (1, 63, 8192, 20_000)]
    off = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
    keys = np.concatenate(parts)
    vals = None if vdt is None else np.arange(keys.size).astype(vdt)
    for desc in (False, True):
        say(f"clusters in segments vals={vdt} desc={desc}")
        tk, tv = dev(keys), None if vals is None else dev(vals)
        handle.sort_segments(tk, dev(off), tv, descending=desc)
        order = np.concatenate([int(a) + stable_order(keys[int(a):int(b)], desc) for a, b in zip(off, off[1:])])
        order = order.astype(np.int64)
        assert_bits_equal(host(tk), keys[order], "keys")
        if vals is not None:
            assert_bits_equal(host(tv), vals[order], "payloads")


def _best_ms(call, prepare) -> float:
    import torch

    ms = []
    for _ in range(4):
        prepare()
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        call()
        t1.record()
        torch.cuda.synchronize()
        ms.append(t0.elapsed_time(t1))
    return min(ms[1:])


@pytest.mark.parametrize("log_n", [22, 24, 26])
def test_clusters_cost_no_multiple(handle, log_n):
    """All digits take about 1.8 times as long as the highest four; a thread a run, or a
    workgroup a run, took up to 40 times as long."""
    import torch

    n = 1 << log_n
    gen = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda lo, hi, m: torch.randint(lo, hi, (m,), generator=gen, device="cuda", dtype=torch.int64)
    wk, wv = torch.empty(n, dtype=torch.uint64, device="cuda"), torch.empty(n, dtype=torch.uint32, device="cuda")
    v = torch.arange(n, device="cuda", dtype=torch.int32).view(torch.uint32)
    ms = {}
    for log_c in (64, 12, 14, 16, 18, 20, 22):
        if log_c == 64:
            k = rand(-(1 << 63), (1 << 63) - 1, n)
        else:
            k = (rand(-(1 << 31), (1 << 31) - 1, 1 << log_c)[rand(0, 1 << log_c, n)] << 32) | rand(0, 1 << 32, n)
        say(f"time of 2^{log_c} clusters, n={n}")
        ms[log_c] = _best_ms(lambda: handle.sort_pairs(wk, wv), lambda: (wk.copy_(k.view(torch.uint64)), wv.copy_(v)))
    print(ms)
    for t in ms.values():
        assert t < 3 * ms[64], ms
