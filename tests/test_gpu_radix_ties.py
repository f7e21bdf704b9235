"""64-bit keys sorted by their highest digits, then put in order where keys
agree in them: pairs and short runs across chunk ends, runs of 31-34 keys
(both sides of the limit between one thread and one workgroup), a run that
fits a workgroup's tile and one that does not, equal keys, constant digits,
and keys whose differences all lie low; single arrays and segments."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu


def planted(n, runs, seed, low_bits=32):
    """Random keys; for every (count, length): `count` groups of `length` keys
    that share all but their lowest bits, a third of those keys equal."""
    r = np.random.RandomState(seed)
    x = r.randint(0, 1 << 63, n, dtype=np.uint64) * np.uint64(2) + r.randint(0, 2, n).astype(np.uint64)
    at = 0
    for count, length in runs:
        for _ in range(count):
            m = x[at:at + length]
            base = m[0] >> np.uint64(low_bits) << np.uint64(low_bits)
            low = m & np.uint64((1 << low_bits) - 1)
            low[r.rand(m.size) < 0.3] = 7
            x[at:at + length] = base | low
            at += length
    assert at <= n
    return x[r.permutation(n)]


CASES = {
    "pairs": (200_003, [(3000, 2), (500, 3), (50, 8)]),
    "limit": (150_001, [(20, 31), (20, 32), (20, 33), (20, 34), (3, 100)]),
    "tile": (260_000, [(1, 5000), (2, 64), (1, 9000)]),
    "past_tile": (700_001, [(1, 20_001), (1, 300)]),
    "uniform": (1 << 18, []),
}


@pytest.mark.parametrize("vdt", [None, np.uint32, np.uint64], ids=lambda t: "none" if t is None else np.dtype(t).name)
@pytest.mark.parametrize("name", sorted(CASES))
def test_planted_runs(handle, name, vdt):
    n, runs = CASES[name]
    keys = planted(n, runs, 7 + len(name))
    for kdt, desc in ((np.uint64, False), (np.int64, True), (np.float64, False)):
        k = keys.view(kdt)
        if kdt is np.float64:  # exponent cleared of infinities and NaNs
            k = (keys & ~np.uint64(1 << 62)).view(kdt)
        vals = None if vdt is None else np.arange(n).astype(vdt)
        order = stable_order(k, desc)
        say(f"ties {name} {np.dtype(kdt).name} vals={vdt} desc={desc}")
        tk, tv = dev(k), None if vals is None else dev(vals)
        if vals is None:
            handle.sort_keys(tk, descending=desc)
        else:
            handle.sort_pairs(tk, tv, descending=desc)
            assert_bits_equal(host(tv), vals[order], f"{name} payloads")
        assert_bits_equal(host(tk), k[order], f"{name} keys")


@pytest.mark.parametrize("vdt", [None, np.uint32, np.uint64], ids=lambda t: "none" if t is None else np.dtype(t).name)
def test_planted_runs_in_segments(handle, vdt):
    parts = [planted(n, runs, 40 + i) for i, (n, runs) in enumerate(CASES.values())]
    parts += [planted(17_000, [(400, 2), (2, 40)], 50), planted(33, [], 51), np.full(30_000, 5, np.uint64)]
    # A segment of equal high digits next to one that starts with them.
    parts += [parts[0][:40_000] >> np.uint64(34), parts[0][:40_000] >> np.uint64(34)]
    off = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
    keys = np.concatenate(parts)
    vals = None if vdt is None else np.arange(keys.size).astype(vdt)
    for chosen in (list(range(len(parts))), list(range(6))):  # with and without the segments that need every digit
        o = np.concatenate([[0], np.cumsum([parts[i].size for i in chosen])]).astype(np.uint64)
        k = np.concatenate([parts[i] for i in chosen])
        v = None if vals is None else vals[:k.size]
        order = np.concatenate([int(o[j]) + stable_order(parts[i]) for j, i in enumerate(chosen)])
        say(f"ties segments vals={vdt} nseg={len(chosen)}")
        tk, tv = dev(k), None if v is None else dev(v)
        handle.sort_segments(tk, dev(o), tv)
        assert_bits_equal(host(tk), k[order], "segment keys")
        if v is not None:
            assert_bits_equal(host(tv), v[order], "segment payloads")


@pytest.mark.parametrize("kind", ["small", "mid_digits", "two_values", "sorted", "pairs_everywhere"])
def test_key_ranges(handle, kind):
    n = 300_007
    r = np.random.RandomState(3)
    x = r.randint(0, 1 << 63, n, dtype=np.uint64)
    k = {"small": x % np.uint64(1000), "mid_digits": (x >> np.uint64(40)) << np.uint64(16),
         "two_values": np.where(x & np.uint64(1), np.uint64(3), np.uint64(1 << 60)), "sorted": np.sort(x),
         "pairs_everywhere": (x[r.randint(0, n // 2, n)] & ~np.uint64(0xFFFF)) | (x & np.uint64(0xFFFF))}[kind]
    v = np.arange(n, dtype=np.uint32)
    order = stable_order(k)
    say(f"ties range {kind}")
    tk, tv = dev(k), dev(v)
    handle.sort_pairs(tk, tv)
    assert_bits_equal(host(tk), k[order], "keys")
    assert_bits_equal(host(tv), v[order], "payloads")
