"""Batches whose long segments make few tiles (smaller tiles and 1024-thread
histograms) and one that does not: lengths at the edges of both tile sizes
(18432 and 28672 keys, 13312 and 19456 pairs), single- and multi-tile segments
side by side, against numpy's stable sort of every segment, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu

EDGES = [16385, 18431, 18432, 18433, 28671, 28672, 28673, 36864, 36865, 57345, 3, 0, 1, 100000]
EDGES_KV = [16385, 13312, 13313, 19455, 19456, 19457, 26624, 26625, 39937, 3, 0, 1, 70001]


@pytest.mark.parametrize("kdt,vdt", [(np.float32, None), (np.int32, np.uint32), (np.uint32, np.int64),
                                     (np.uint64, None)], ids=lambda t: "none" if t is None else np.dtype(t).name)
@pytest.mark.parametrize("desc", [False, True], ids=["asc", "desc"])
@pytest.mark.parametrize("repeat", [1, 3, 20])  # 20: more tiles than two rounds of CUs
def test_segments_at_tile_edges(handle, kdt, vdt, desc, repeat):
    lengths = (EDGES if vdt is None else EDGES_KV) * repeat
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    n = int(off[-1])
    rng = np.random.RandomState(repeat)
    keys = rng.randn(n).astype(kdt) if np.dtype(kdt).kind == "f" else rng.randint(0, 2**31, n).astype(kdt)
    order = np.concatenate([int(a) + stable_order(keys[int(a):int(b)], desc) for a, b in zip(off, off[1:])])
    order = order.astype(np.int64)
    tk, to = dev(keys), dev(off.view(np.int64))
    say(f"segments {np.dtype(kdt)} {vdt} desc={desc} x{repeat} n={n}")
    import torch

    if vdt is None:
        handle.sort_segments(tk, to.view(torch.uint64), descending=desc)
    else:
        tv = dev(np.arange(n).astype(vdt))
        handle.sort_segments(tk, to.view(torch.uint64), tv, descending=desc)
        assert_bits_equal(host(tv), order.astype(vdt), "payloads")
    assert_bits_equal(host(tk), keys[order], "keys")
