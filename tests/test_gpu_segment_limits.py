"""small_max of a batched sort's size classes decides which kernels sort the
segments past it, with and without a medium class: at its limit the LDS tile,
below it the radix passes (their histogram shows in the profile)."""
from __future__ import annotations

import numpy as np
import pytest
from gpu_util import assert_bits_equal, dev, host, say, stable_order
from gpusort_amd import I64, NONE, U32, U64

pytestmark = pytest.mark.gpu

TYPES = {U32: np.uint32, U64: np.uint64, I64: np.int64}


@pytest.mark.parametrize("kdt,vdt,limit", [(U32, NONE, 8192), (U32, U32, 4096), (U64, U32, 2048), (I64, I64, 2048)])
@pytest.mark.parametrize("medium_max", [0, 700])
def test_small_max_decides(handle, kdt, vdt, limit, medium_max):
    lengths = [2001, 3, 1999, 0, 1024, 1025, 600, 701, 2000] * 20
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint64)
    n = int(off[-1])
    keys = np.random.RandomState(n).randint(0, 1 << 31, n).astype(TYPES[kdt])
    vals = None if vdt == NONE else np.arange(n).astype(TYPES[vdt])
    order = np.concatenate([int(a) + stable_order(keys[int(a):int(b)]) for a, b in zip(off, off[1:])]).astype(np.int64)
    before = handle.seg_config(kdt, vdt)
    try:
        for small_max, passes in ((limit, medium_max > 0 and small_max_below(limit, lengths, medium_max)),
                                  (1024, True), (512, True)):
            handle.set_seg_config(kdt, vdt, small_max, medium_max)
            say(f"segments with small_max={small_max} medium_max={medium_max}")
            tk, tv = dev(keys), None if vals is None else dev(vals)
            handle.profile_begin()
            handle.sort_segments(tk, dev(off), tv)
            assert ("seg_hist" in handle.profile_end()) == passes, (small_max, medium_max)
            assert_bits_equal(host(tk), keys[order], "keys")
            if vals is not None:
                assert_bits_equal(host(tv), vals[order], "payloads")
    finally:
        handle.set_seg_config(kdt, vdt, before["small_max"], before["medium_max"], before["medium_geometry"])


def small_max_below(limit, lengths, medium_max) -> bool:
    """Whether a segment is past the LDS limit and in the medium class."""
    return any(limit < m <= medium_max for m in lengths)
