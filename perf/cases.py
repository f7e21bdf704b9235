"""Timed workloads of the sort library: what its callers have it do, each
through a public entry point of ``gpusort_amd``.

A case is a dict of plain values; ``prepare`` makes its inputs on the device
(or, for the host-memory sort, on the host), ``run`` is one call as a caller
makes it, ``work`` the bytes that call cannot do without.  The sorts work in
place, so ``run`` first copies the kept input into the array to be sorted, as
a caller that still needs its input does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import gpusort_amd as g

# name -> (element bytes, dtype the library is given, dtype torch computes in)
_TYPES = {
    "i32": (4, torch.int32, torch.int32),
    "u32": (4, torch.uint32, torch.int32),
    "f32": (4, torch.float32, torch.float32),
    "i64": (8, torch.int64, torch.int64),
    "u64": (8, torch.uint64, torch.int64),
    "f64": (8, torch.float64, torch.float64),
}
_ALGORITHMS = {"hyksort": g.HYKSORT, "samplesort": g.SAMPLESORT, "hyperquicksort": g.HYPERQUICKSORT}


def listed() -> list[dict]:
    return [
        # The smallest call: one workgroup's worth of pairs, all latency.
        {"name": "pairs_1k", "kind": "sort", "key": "u32", "val": "u32", "n": 1000, "dist": "uniform", "desc": False},
        # An ordinary odd-sized array of measurements with their indexes, largest first.
        {"name": "pairs_1m_f32", "kind": "sort", "key": "f32", "val": "u32", "n": 1_000_003, "dist": "uniform",
         "desc": True},
        # One rank's local sort of keys alone (the single-rank configuration of the benchmark).
        {"name": "keys_16m", "kind": "sort", "key": "u32", "val": "", "n": 1 << 24, "dist": "uniform", "desc": False},
        # Double keys with 64-bit payloads: the widest element.
        {"name": "pairs_32m_f64", "kind": "sort", "key": "f64", "val": "i64", "n": (1 << 25) + 35, "dist": "uniform",
         "desc": False},
        # The benchmark's headline: a large stable key-value sort.
        {"name": "pairs_256m", "kind": "sort", "key": "u32", "val": "u32", "n": 1 << 28, "dist": "uniform",
         "desc": False},
        # Many arrays of very different lengths sorted by one call.
        {"name": "batch_20k", "kind": "batch", "key": "u32", "val": "u32", "arrays": 20_000, "median": 2048,
         "sigma": 2.0, "desc": False},
        # HykSort over 64 ranks of 2^21 keys with original indexes (local sort, splitters, k-way merges).
        {"name": "hyksort_64", "kind": "ranks", "algo": "hyksort", "key": "u64", "val": "u32", "p": 64,
         "per_rank": 1 << 21, "ragged": False, "k": 8, "desc": False},
        # SampleSort over 16 ranks of unequal sizes, keys alone.
        {"name": "samplesort_16", "kind": "ranks", "algo": "samplesort", "key": "f32", "val": "", "p": 16,
         "per_rank": 250_007, "ragged": True, "k": 8, "desc": False},
        # Unsorted pairs cut into one bucket per receiving rank.
        {"name": "multisplit_64", "kind": "multisplit", "key": "u32", "val": "u32", "n": 1 << 28, "buckets": 64},
        # Two sorted runs of unequal length merged (the last step of a chunked sort).
        {"name": "merge_50m", "kind": "merge", "key": "u32", "val": "u32", "na": (1 << 25) + 7, "nb": (1 << 24) + 999,
         "desc": False},
        # Several payload vectors: sort keys with a global index, then gather each vector by it.
        {"name": "global_index_128m", "kind": "index", "key": "u32", "n": 1 << 27},
        # Host vectors in, host vectors out (the local-sort seam as host code calls it).
        {"name": "host_pairs_1m", "kind": "host", "key": "u32", "val": "u32", "n": 1_000_003, "desc": False},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["sort", "sort", "sort", "batch", "ranks", "multisplit", "merge", "index", "host"])
    key = rng.choice(sorted(_TYPES))
    val = rng.choice(["", "u32", "u32", "i64"])
    desc = rng.random() < 0.3
    width = _TYPES[key][0] + (_TYPES[val][0] if val else 0)
    if kind == "sort":
        return {"kind": kind, "key": key, "val": val, "n": _log_int(rng, 200, (1 << 31) // width),
                "dist": rng.choice(["uniform", "uniform", "zipf", "sorted"]), "desc": desc}
    if kind == "batch":
        return {"kind": kind, "key": key, "val": val, "arrays": _log_int(rng, 50, 20_000),
                "median": _log_int(rng, 100, 2048), "sigma": round(rng.uniform(0.5, 2.0), 3), "desc": desc}
    if kind == "ranks":
        p = rng.choice([4, 8, 16, 32, 64])
        return {"kind": kind, "algo": rng.choice(sorted(_ALGORITHMS)), "key": key, "val": rng.choice(["", "u32"]),
                "p": p, "per_rank": _log_int(rng, 5000, (1 << 26) // p), "ragged": rng.random() < 0.5,
                "k": rng.choice([2, 4, 8]), "desc": desc}
    if kind == "multisplit":
        return {"kind": kind, "key": key, "val": val, "n": _log_int(rng, 50_000, (1 << 31) // width),
                "buckets": rng.choice([2, 8, 31, 64, 200, 256])}
    if kind == "merge":
        return {"kind": kind, "key": key, "val": val, "na": _log_int(rng, 1000, 1 << 25),
                "nb": _log_int(rng, 1000, 1 << 25), "desc": desc}
    if kind == "index":
        return {"kind": kind, "key": rng.choice(["u32", "i32", "f32", "u64"]), "n": _log_int(rng, 50_000, 1 << 26)}
    return {"kind": "host", "key": key, "val": val or "u32", "n": _log_int(rng, 1000, 1 << 22), "desc": desc}


# ------------------------------------------------------------------ inputs

_handle: g.Handle | None = None


def _lib() -> g.Handle:
    """The one handle (device, null stream, workspace) a program keeps."""
    global _handle
    if _handle is None:
        _handle = g.Handle()
    return _handle


def _keys(name: str, n: int, dist: str, seed: int) -> torch.Tensor:
    """n keys of type `name` in torch's compute dtype: all bit patterns of the
    integers, N(0, 1000) floats without -0.0, or few heavy values (zipf) / an
    array already in order (sorted)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    size, _, dt = _TYPES[name]
    is_float = dt.is_floating_point
    if dist == "zipf":
        # Zipf(1.1) ranks of 2^20 values by the inverse of the continuous law, spread by an odd multiplier.
        u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
        rank = (1.0 - u * (1.0 - float(1 << 20) ** -0.1)).pow_(-10.0).floor_().to(torch.int64)
        if is_float:
            return rank.to(dt)
        x = rank * (0x9E3779B97F4A7C15 - (1 << 64))
        return x if size == 8 else (x >> 32).to(torch.int32)
    if is_float:
        x = torch.randn(n, generator=gen, device="cuda", dtype=dt).mul_(1e3).add_(0.0)
    else:
        bits = size * 8 - 1
        x = torch.randint(-(1 << bits), (1 << bits) - 1, (n,), generator=gen, device="cuda", dtype=dt)
    return torch.sort(x)[0] if dist == "sorted" else x


def _payload(name: str, n: int) -> torch.Tensor | None:
    """Original positions, the payload the library's callers carry."""
    return torch.arange(n, device="cuda", dtype=_TYPES[name][2]) if name else None


def _typed(t: torch.Tensor | None, name: str) -> torch.Tensor | None:
    return None if t is None else t.view(_TYPES[name][1])


def _lengths(case: dict, seed: int) -> np.ndarray:
    """Array lengths at the lognormal law's own quantiles (one total for every
    seed), in an order drawn from the seed."""
    m = case["arrays"]
    q = (torch.arange(m, dtype=torch.float64) + 0.5) / m
    length = (math.log(case["median"]) + case["sigma"] * torch.special.ndtri(q)).exp().round().clamp(1, 1 << 22)
    return length.numpy().astype(np.int64)[np.random.RandomState(seed % (1 << 32)).permutation(m)]


def _rank_sizes(case: dict, seed: int) -> np.ndarray:
    p, per = case["p"], case["per_rank"]
    if not case["ragged"]:
        return np.full(p, per, dtype=np.int64)
    size = (np.linspace(0.4, 1.6, p) * per).astype(np.int64)
    return size[np.random.RandomState(seed % (1 << 32)).permutation(p)]


def _offsets(sizes: np.ndarray) -> np.ndarray:
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = {"case": case, "h": _lib()}
    key, val = case["key"], case.get("val", "")
    if kind == "merge":
        for side, n in (("a", case["na"]), ("b", case["nb"])):
            k = torch.sort(_keys(key, n, "uniform", 2 * seed + (side == "b")), descending=False)[0]
            if key in ("u32", "u64"):  # unsigned order: the halves of the signed order swapped
                k = torch.cat([k[k >= 0], k[k < 0]])
            s[side + "k"] = k.flip(0).contiguous() if case["desc"] else k
            s[side + "v"] = _payload(val, n)
        n = case["na"] + case["nb"]
        s["ok"] = torch.empty(n, device="cuda", dtype=_TYPES[key][2])
        s["ov"] = torch.empty(n, device="cuda", dtype=_TYPES[val][2]) if val else None
        return s
    if kind == "batch":
        off = _offsets(_lengths(case, seed))
        n = int(off[-1])
        s["off"] = torch.from_numpy(off.view(np.int64)).to("cuda").view(torch.uint64)
    elif kind == "ranks":
        s["off"] = _offsets(_rank_sizes(case, seed))
        n = int(s["off"][-1])
    else:
        n = case["n"]
    k = _keys(key, n, case.get("dist", "uniform"), seed)
    v = _payload(val, n)
    if kind == "host":
        s["k"], s["v"] = k.cpu().numpy(), v.cpu().numpy()
        s["wk"], s["wv"] = np.empty_like(s["k"]), np.empty_like(s["v"])
        return s
    s["k"], s["v"] = k, v
    s["wk"], s["wv"] = torch.empty_like(k), None if v is None else torch.empty_like(v)
    if kind == "multisplit":
        # Regular samples of the keys, in the library's (unsigned, signed or float) order.
        sample = k[:: max(1, n // 8192)].cpu().numpy()
        sample = np.sort(sample.view({"u32": np.uint32, "u64": np.uint64}.get(key, sample.dtype)))
        b = case["buckets"]
        s["spl"] = sample[(np.arange(1, b) * sample.size) // b]
    elif kind == "index":
        gen = torch.Generator(device="cuda").manual_seed(seed + 1)
        s["pay"] = [torch.randint(-(1 << 31), (1 << 31) - 1, (n,), generator=gen, device="cuda", dtype=torch.int32),
                    torch.rand(n, generator=gen, device="cuda", dtype=torch.float64),
                    torch.randint(-(1 << 15), (1 << 15) - 1, (n,), generator=gen, device="cuda", dtype=torch.int16)]
        s["out"] = [torch.empty_like(x) for x in s["pay"]]
        s["idx"] = torch.empty(n, device="cuda", dtype=torch.int64)
    return s


# ------------------------------------------------------------------ one pass


def run(s: dict):
    case, h = s["case"], s["h"]
    kind, key, val = case["kind"], case["key"], case.get("val", "")
    if kind == "merge":
        h.merge(_typed(s["ak"], key), _typed(s["bk"], key), _typed(s["ok"], key), _typed(s["av"], val),
                _typed(s["bv"], val), _typed(s["ov"], val), descending=case["desc"])
        return [s["ok"]] if s["ov"] is None else [s["ok"], s["ov"]]
    if kind == "multisplit":
        off = h.multisplit(_typed(s["k"], key), s["spl"], _typed(s["wk"], key), _typed(s["v"], val),
                           _typed(s["wv"], val))
        out = [s["wk"]] if s["wv"] is None else [s["wk"], s["wv"]]
        return out + [off.view(np.int64)]
    if kind == "host":
        np.copyto(s["wk"], s["k"])
        np.copyto(s["wv"], s["v"])
        as_np = {"u32": np.uint32, "u64": np.uint64}
        h.sort_pairs_host(s["wk"].view(as_np.get(key, s["wk"].dtype)), s["wv"].view(as_np.get(val, s["wv"].dtype)),
                          descending=case["desc"])
        return [s["wk"], s["wv"]]
    wk = _typed(s["wk"], key)
    s["wk"].copy_(s["k"])
    if kind == "index":
        torch.arange(case["n"], out=s["idx"])
        h.sort_pairs(wk, s["idx"])
        for src, dst in zip(s["pay"], s["out"]):
            h.gather(src, s["idx"], dst)
        return [s["wk"], s["idx"], *s["out"]]
    wv = _typed(s["wv"], val)
    if wv is not None:
        s["wv"].copy_(s["v"])
    out = [s["wk"]] if wv is None else [s["wk"], s["wv"]]
    if kind == "batch":
        h.sort_segments(wk, s["off"], wv, descending=case["desc"])
    elif kind == "ranks":
        rep = h.vrank_sort(wk, s["off"], wv, algorithm=_ALGORITHMS[case["algo"]], k_way=case["k"],
                           samples_per_rank=32, descending=case["desc"])
        spl = rep["splitters"]
        out = out + [spl if spl.dtype.kind == "f" else spl.view(f"i{spl.itemsize}"),
                     rep["bucket_sizes"].view(np.int64), rep["final_rank_sizes"].view(np.int64)]
    elif wv is None:
        h.sort_keys(wk, descending=case["desc"])
    else:
        h.sort_pairs(wk, wv, descending=case["desc"])
    return out


# ------------------------------------------------------------------ what a pass needs


def work(case: dict) -> dict:
    """Every key and payload read once and written once (for the global index:
    the keys, the index written, and each payload vector)."""
    kind = case["kind"]
    kb = _TYPES[case["key"]][0]
    vb = _TYPES[case["val"]][0] if case.get("val") else 0
    if kind == "index":
        return {"bytes": case["n"] * (2 * kb + 8 + 2 * (4 + 8 + 2)), "flops": 0}
    if kind == "merge":
        n = case["na"] + case["nb"]
    elif kind == "batch":
        n = int(_lengths(case, 0).sum())
    elif kind == "ranks":
        n = int(_rank_sizes(case, 0).sum())
    else:
        n = case["n"]
    return {"bytes": 2 * n * (kb + vb), "flops": 0}


def exact(case: dict, seed: int):
    """Outputs are the inputs rearranged; where they are floating point, the
    same rearrangement by torch's stable sort (the others are whole numbers)."""
    kind, key = case["kind"], case["key"]
    if kind == "index":
        s = prepare(case, seed)
        k = s["k"].long() & 0xFFFFFFFF if key == "u32" else s["k"] ^ (-1 << 63) if key == "u64" else s["k"]
        order = torch.sort(k, stable=True)[1]
        keys = s["k"][order].double() if key.startswith("f") else None
        return [keys, None, None, s["pay"][1][order], None]
    if not key.startswith("f") or kind not in ("sort", "host", "ranks", "merge"):
        return None
    val = case["val"]
    if kind == "merge":
        s = prepare(case, seed)
        k = torch.cat([s["ak"], s["bk"]])
    else:
        n = int(_rank_sizes(case, seed).sum()) if kind == "ranks" else case["n"]
        k = _keys(key, n, case.get("dist", "uniform"), seed)
    k = torch.sort(k.double(), descending=case["desc"])[0]
    return [k] + [None] * ((3 if kind == "ranks" else 0) + bool(val))
