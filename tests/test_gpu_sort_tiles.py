"""Single-array radix sorts around the sizes where the tile changes (and one
past a whole number of tiles), with keys of which one, two or three digits vary
(an odd number: one of the passes left out copies the result home) and with all
of them varying, against numpy's stable sort, bit for bit.  The fixed scratch
of the no-allocation entry takes the sizes that it took with the largest tiles."""
from __future__ import annotations

import numpy as np
import pytest
from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu

TYPES = [(np.uint32, None), (np.float32, np.uint32), (np.uint32, np.int64), (np.uint64, None), (np.int64, np.uint32),
         (np.uint64, np.int64)]


def _keys(dt, n: int, digits: int) -> np.ndarray:
    rng = np.random.RandomState(n % 1000 + digits)
    size = np.dtype(dt).itemsize
    bits = rng.randint(0, 2**32, n).astype(np.uint64) | (rng.randint(0, 2**32, n).astype(np.uint64) << np.uint64(32))
    # The lowest byte and, from three digits on, the highest ones vary.
    at = [0, size - 2, 1][:digits] if digits < 4 else range(size)
    mask = np.uint64(sum(0xFF << (8 * b) for b in at))
    raw = (bits & mask).astype(np.uint64 if size == 8 else np.uint32)
    if np.dtype(dt).kind == "f" and digits >= 4:
        return rng.randn(n).astype(dt) + dt(0)
    return raw.view(dt)


@pytest.mark.parametrize("kdt,vdt", TYPES, ids=lambda t: "none" if t is None else np.dtype(t).name)
@pytest.mark.parametrize("n", [16385, 20480 * 3 + 1, (1 << 18) + 1, 3 << 17, (3 << 17) + 1, (1 << 19) + 1, 1 << 20,
                               (1 << 20) + 1, 256 * 1024 * 10, 256 * 1024 * 10 + 1, 256 * 1024 * 22 + 1])
def test_sorts_around_the_tile_rules(handle, kdt, vdt, n):
    for digits in (1, 2, 3, 8):
        keys = _keys(kdt, n, digits)
        desc = digits == 2
        order = stable_order(keys, desc)
        tk = dev(keys)
        say(f"sort {np.dtype(kdt)} {vdt} n={n} digits={digits} desc={desc}")
        if vdt is None:
            handle.sort_keys(tk, descending=desc)
        else:
            tv = dev(np.arange(n).astype(vdt))
            handle.sort_pairs(tk, tv, descending=desc)
            assert_bits_equal(host(tv), order.astype(vdt), f"payloads {digits}")
        assert_bits_equal(host(tk), keys[order], f"keys {digits}")


def test_scratch_limit_is_the_large_tiles(handle):
    """18.2 M u32 keys fit the 72 MiB scratch with tiles of 30 items only."""
    n = 18_200_000
    keys = _keys(np.uint32, n, 8)
    tk = dev(keys)
    say("no-allocation sort at its limit")
    handle.sort_pairs_noalloc(tk, None)
    assert_bits_equal(host(tk), np.sort(keys), "keys")
