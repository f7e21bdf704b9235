"""64-bit keys of which many share their high digits (a sentinel with a few small
numbers, small ids or a hot prefix among random keys): runs that no workgroup's
tile holds are sorted by all workgroups together, one digit after another, and
never cost many times what other keys of the same number do.  One to four of the
lowest digits vary (an odd and an even number of moves), chunks of a run end in
the middle, several runs differ in the digits that vary, and runs below and above
the tile stand side by side."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu


_SENTINELS = {"sentinel1": 0xF, "sentinel2": 0xFF00FF, "sentinel3": 0xF0F00F}


def _random(r, n):
    return r.randint(0, 1 << 63, n, dtype=np.uint64) * np.uint64(2) + r.randint(0, 2, n).astype(np.uint64)


def _keys(name: str, n: int, seed: int) -> np.ndarray:
    r = np.random.RandomState(seed)
    x = _random(r, n)
    if name == "uniform":
        return x
    if name == "hot":  # one key in twenty shares its upper half
        m = r.rand(n) < 0.05
        x[m] = (x[m] & np.uint64(0xFFFFFFFF)) | np.uint64(77 << 32)
        return x
    if name == "small":  # half the keys are small numbers
        m = r.rand(n) < 0.5
        x[m] %= np.uint64(100)
        return x
    if name in _SENTINELS:  # half the keys equal, a few others close to them
        m = np.nonzero(r.rand(n) < 0.5)[0]
        x[m] = 0
        few = r.choice(m, 24, replace=False)
        x[few] = _random(r, 24) & np.uint64(_SENTINELS[name])
        return x
    if name == "sentinels":  # three such runs of very different lengths
        u = r.rand(n)
        for j, (lo, hi, mask) in enumerate([(0.0, 0.4, 0xFF00), (0.4, 0.42, 0xFFFFFFFF), (0.42, 0.65, 0xF0F)]):
            m = np.nonzero((u >= lo) & (u < hi))[0]
            x[m] = (j + 5) << 33
            few = r.choice(m, 24, replace=False)
            x[few] += _random(r, 24) & np.uint64(mask)
        return x
    if name == "several":  # runs of 5000 to 30,000 keys that vary in different digits
        at = 0
        for j, size in enumerate([5000, 30_000, 12_288, 12_289, 8192, 8193, 20_480, 6145, 16_385]):
            mask = sum(0xFF << (8 * d) for d in range(4) if (j + 1) >> (d % 4) & 1 or j == 1)
            x[at:at + size] = (x[at:at + size] & np.uint64(mask)) | np.uint64((1000 + j) << 32)
            at += size
        return x[r.permutation(n)]
    raise ValueError(name)


CASES = [("hot", (1 << 23) + 5), ("several", (1 << 23) + 11), ("hot", 1 << 20), ("sentinel1", 1 << 18), ("sentinel2", (1 << 18) + 4097),
         ("sentinel3", 300_001), ("small", 200_003), ("sentinel2", (1 << 22) + 9), ("sentinels", 5_000_011)]


@pytest.mark.parametrize("vdt", [None, np.uint32, np.uint64], ids=lambda t: "none" if t is None else np.dtype(t).name)
@pytest.mark.parametrize("name,n", CASES)
def test_runs_past_a_tile(handle, name, n, vdt):
    keys = _keys(name, n, n)
    for kdt, desc in ((np.uint64, False), (np.int64, True)):
        k = keys.view(kdt)
        vals = None if vdt is None else np.arange(n).astype(vdt)
        order = stable_order(k, desc)
        say(f"runs {name} {np.dtype(kdt).name} n={n} vals={vdt} desc={desc}")
        tk, tv = dev(k), None if vals is None else dev(vals)
        if vals is None:
            handle.sort_keys(tk, descending=desc)
        else:
            handle.sort_pairs(tk, tv, descending=desc)
            assert_bits_equal(host(tv), vals[order], f"{name} payloads")
        assert_bits_equal(host(tk), k[order], f"{name} keys")


@pytest.mark.parametrize("vdt", [None, np.uint32, np.uint64], ids=lambda t: "none" if t is None else np.dtype(t).name)
def test_runs_in_segments(handle, vdt):
    parts = [_keys("several", (1 << 23) + 3, 1), _keys("uniform", 20_000, 2), _keys("hot", 1 << 23, 3),
             _keys("uniform", 13_000, 4), _keys("sentinel3", 120_001, 5), _keys("uniform", 777, 6)]
    off = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
    keys = np.concatenate(parts)
    vals = None if vdt is None else np.arange(keys.size).astype(vdt)
    for desc in (False, True):
        say(f"runs in segments vals={vdt} desc={desc}")
        tk, tv = dev(keys), None if vals is None else dev(vals)
        handle.sort_segments(tk, dev(off), tv, descending=desc)
        gk, gv = host(tk), None if vals is None else host(tv)
        for a, b in zip(off[:-1].astype(int), off[1:].astype(int)):
            order = stable_order(keys[a:b], desc)
            assert_bits_equal(gk[a:b], keys[a:b][order], f"keys of [{a}, {b})")
            if vals is not None:
                assert_bits_equal(gv[a:b], vals[a:b][order], f"payloads of [{a}, {b})")


def test_runs_in_a_graph_and_without_allocation(handle):
    """A plan's captured graph replayed between eager sorts (the tasks' counters start
    from zero every time), and the entry whose workspace is a fixed array."""
    import torch
    from gpusort_amd import U32, U64

    parts = [_keys("sentinel3", 400_003, 5), _keys("uniform", 30_000, 6), _keys("sentinels", 300_000, 7)]
    off = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
    keys = np.concatenate(parts)
    vals = np.arange(keys.size, dtype=np.uint32)
    order = np.concatenate([int(a) + stable_order(keys[int(a):int(b)]) for a, b in zip(off, off[1:])]).astype(np.int64)
    k0, v0 = dev(keys), dev(vals)
    tk, tv = k0.clone(), v0.clone()
    torch.cuda.synchronize()
    plan = handle.seg_plan(off, U64, U32)
    try:
        for replay in range(4):
            tk.copy_(k0)
            tv.copy_(v0)
            torch.cuda.synchronize()
            say(f"runs in a graph, replay {replay}")
            plan.launch_graph(tk, tv)
            torch.cuda.synchronize()
            assert_bits_equal(host(tk), keys[order], "keys")
            assert_bits_equal(host(tv), vals[order], "payloads")
            ek = dev(parts[0])
            handle.sort_keys(ek)
            assert_bits_equal(host(ek), np.sort(parts[0]), "eager keys")
    finally:
        plan.close()
    one = parts[0]
    tk, tv = dev(one), dev(np.arange(one.size, dtype=np.uint32))
    say("runs without allocation")
    assert handle.lib.gs_sort_pairs_noalloc(handle.h, U64, tk.data_ptr(), U32, tv.data_ptr(), one.size, 0) == 0
    torch.cuda.synchronize()
    assert_bits_equal(host(tv), stable_order(one).astype(np.uint32), "payloads")


def test_runs_on_several_streams_at_once():
    """Handles on streams of their own sort at the same time, each with runs that its
    workgroups share: no sort waits for another one's workgroups."""
    import torch
    import gpusort_amd

    n, m = 500_009, 4
    keys = [_keys(("sentinels", "sentinel3", "sentinel1", "sentinel2")[i], n + i, i) for i in range(m)]
    streams = [torch.cuda.Stream() for _ in range(m)]
    handles = [gpusort_amd.Handle(0, stream=s) for s in streams]
    base = [dev(k) for k in keys]
    work = [[b.clone() for b in base] for _ in range(6)]
    torch.cuda.synchronize()
    say("runs on several streams")
    for turn in work:
        for h, w in zip(handles, turn):
            h.sort_keys(w)
    torch.cuda.synchronize()
    for turn in work:
        for w, k in zip(turn, keys):
            assert_bits_equal(host(w), np.sort(k), "keys")
    for h in handles:
        h.close()


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


def test_keys_that_share_a_prefix_cost_no_multiple(handle):
    """At 2^24 pairs all digits take about 1.8 times as long as the highest four; one
    workgroup alone with a twentieth of the keys took 20 times as long."""
    import torch

    n = 1 << 24
    wk, wv = torch.empty(n, dtype=torch.uint64, device="cuda"), torch.empty(n, dtype=torch.uint32, device="cuda")
    ms = {}
    for name in ("uniform", "hot", "small", "sentinel1", "sentinel2"):
        k, v = dev(_keys(name, n, 9)), torch.arange(n, dtype=torch.int32, device="cuda").view(torch.uint32)
        say(f"time of {name}")
        ms[name] = _best_ms(lambda: handle.sort_pairs(wk, wv), lambda: (wk.copy_(k), wv.copy_(v)))
    print(ms)
    for name, t in ms.items():
        assert t < 4 * ms["uniform"], ms


def test_runs_of_a_large_array(handle):
    """2^30 keys and more: positions past 32 bits of status word, counts of 64 bits."""
    import torch

    n = (1 << 30) + 77
    gen = torch.Generator(device="cuda").manual_seed(11)
    k = torch.randint(-(1 << 63), (1 << 63) - 1, (n,), generator=gen, device="cuda", dtype=torch.int64)
    k[: n // 8] = 3 << 40
    k[torch.arange(40, device="cuda") * 1_000_003 + 17] += torch.arange(40, device="cuda") * 0x01010101
    v = torch.arange(n, device="cuda", dtype=torch.int32)
    wk, wv = k.clone(), v.clone()
    say(f"runs of a large array n={n}")
    handle.sort_pairs(wk, wv.view(torch.uint32))
    for at in range(0, n - 1, 1 << 27):
        end = min(n, at + (1 << 27) + 1)
        a, p = wk[at:end], wv[at:end].long()
        assert torch.equal(k[p], a), "payloads lead to their keys"
        d = (a[:-1] < a[1:]) | ((a[:-1] == a[1:]) & (p[:-1] < p[1:]))
        assert bool(d.all()), "in order, ties by input position (so every position once)"


def test_small_ids_in_late_segments_cost_no_multiple(handle):
    """2300 segments, the last 250 of them small ids: they have a say in the digits
    sorted by like the first."""
    import torch

    m, per = 2300, 14_000
    off = dev(np.arange(m + 1, dtype=np.uint64) * np.uint64(per))
    wk = torch.empty(m * per, dtype=torch.uint64, device="cuda")
    wv = torch.empty(m * per, dtype=torch.uint32, device="cuda")
    x = _keys("uniform", m * per, 4)
    ms = []
    for late in (False, True):
        if late:
            x[2050 * per:] %= np.uint64(1 << 31)
        k, v = dev(x), torch.arange(m * per, dtype=torch.int32, device="cuda").view(torch.uint32)
        say(f"late segments of small ids: {late}")
        ms.append(_best_ms(lambda: handle.sort_segments(wk, off, wv), lambda: (wk.copy_(k), wv.copy_(v))))
    print(ms)
    assert ms[1] < 3 * ms[0], ms
