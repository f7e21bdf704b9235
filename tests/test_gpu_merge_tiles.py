"""2-way merges at the edges of the merge kernel's tiles (6656 elements, 4608
where key and payload take 16 bytes) and of its sixteen-lane split search:
lengths around a tile and around powers of 17, an empty run, runs that do not
interleave, runs of ties, and the key type's largest value, against numpy's
stable sort of the concatenation, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu

SIZES = [(0, 1), (1, 0), (1, 1), (16, 17), (289, 4913), (4607, 1), (0, 4608), (4608, 1), (6655, 1), (1, 6655),
         (6656, 6657), (83521, 3), (3, 83521), (100003, 70001)]


def _runs(kind: str, dt, na: int, nb: int):
    rng = np.random.RandomState(na * 7 + nb)
    top = np.iinfo(dt).max
    if kind == "ties":
        return rng.randint(0, 3, na).astype(dt), rng.randint(0, 3, nb).astype(dt)
    if kind == "apart":
        return np.full(na, top, dt), rng.randint(0, 9, nb).astype(dt)
    a, b = (rng.randint(0, 2**62, n).astype(np.uint64).astype(dt) for n in (na, nb))
    a[: na // 50] = top
    b[: nb // 50] = top
    return a, b


@pytest.mark.parametrize("kdt,vdt", [(np.uint32, None), (np.uint32, np.uint32), (np.int64, np.uint32),
                                     (np.uint64, np.int64)], ids=["u32", "u32-u32", "i64-u32", "u64-i64"])
@pytest.mark.parametrize("kind", ["random", "ties", "apart"])
@pytest.mark.parametrize("desc", [False, True], ids=["asc", "desc"])
def test_merge_at_tile_edges(handle, kdt, vdt, kind, desc):
    for na, nb in SIZES:
        a, b = _runs(kind, kdt, na, nb)
        a, b = a[stable_order(a, desc)], b[stable_order(b, desc)]
        cat = np.concatenate([a, b])
        order = stable_order(cat, desc)
        ok = dev(np.zeros(na + nb, dtype=kdt))
        say(f"merge {np.dtype(kdt)} {vdt} {kind} desc={desc} {na}+{nb}")
        if vdt is None:
            handle.merge(dev(a), dev(b), ok, descending=desc)
        else:
            v = np.arange(na + nb).astype(vdt)
            ov = dev(np.zeros(na + nb, dtype=vdt))
            handle.merge(dev(a), dev(b), ok, dev(v[:na]), dev(v[na:]), ov, descending=desc)
            assert_bits_equal(host(ov), v[order], f"payloads {na}+{nb}")
        assert_bits_equal(host(ok), cat[order], f"keys {na}+{nb}")
