"""The profile of a 64-bit sort counts the passes that ran, with their bytes, and
the two kernels after them by themselves."""
from __future__ import annotations

import numpy as np
import pytest
from gpu_util import dev, say

pytestmark = pytest.mark.gpu


def _random(n, seed):
    r = np.random.RandomState(seed)
    return r.randint(0, 1 << 63, n, dtype=np.uint64) * np.uint64(2) + r.randint(0, 2, n).astype(np.uint64)


@pytest.mark.parametrize("n,digits,passes,ties", [
    (1 << 21, 8, 4, True),     # random keys: the highest four digits
    (1 << 21, 3, 4, False),    # three digits vary: their passes and the one that copies
    (1 << 21, 2, 2, False),    # two
    (1 << 15, 1, 2, False)])
def test_passes_that_ran(handle, n, digits, passes, ties):
    keys = _random(n, n + digits) & np.uint64((1 << (8 * digits)) - 1) << np.uint64(64 - 8 * digits)
    tv = dev(np.arange(n, dtype=np.uint32))
    say(f"profile n={n} digits={digits}")
    handle.profile_begin()
    for _ in range(3):
        handle.sort_pairs(dev(keys), tv)
    p = handle.profile_end()
    assert p["onesweep_pass"]["launches"] == 3 * passes
    assert p["onesweep_pass"]["bytes"] == 3 * passes * 2 * n * 12
    assert ("tie_fix" in p) == ties and ("long_run" in p) == ties
    if ties:
        assert p["tie_fix"]["launches"] == 3 and p["tie_fix"]["bytes"] == 3 * n * 8
        assert p["long_run"]["launches"] == 3


def test_passes_of_segments_that_ran(handle):
    n = 1 << 20
    off = np.array([0, n // 2, n], dtype=np.uint64)
    for mask, passes in ((~np.uint64(0), 4), (np.uint64(0xFFFFFFFF), 8)):
        tk = dev(_random(n, 5) & mask)
        say("profile of segments")
        handle.profile_begin()
        handle.sort_segments(tk, dev(off))
        p = handle.profile_end()
        assert p["seg_onesweep_pass"]["launches"] == passes
        assert p["seg_onesweep_pass"]["bytes"] == passes * 2 * n * 8
        assert ("tie_fix" in p) == (passes == 4)
