"""The one-workgroup sort at the edges of its length classes (single arrays
and segments of one batch), with keys that take each of its paths: differing
bits that fit its first digits, short runs of keys equal in them, long runs
out of order below them (the whole range sorted again), equal keys."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import assert_bits_equal, dev, host, say, stable_order

pytestmark = pytest.mark.gpu

LENGTHS = [2, 63, 64, 65, 255, 256, 257, 1000, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 9215, 9216, 9217,
           12287, 12288, 12289, 16383, 16384, 16385]
TYPES = [(np.uint32, None), (np.int32, np.uint32), (np.float32, np.uint64), (np.uint64, None), (np.int64, np.uint32),
         (np.float64, np.uint64)]


def make(kdt, n, kind, seed):
    d = np.dtype(kdt)
    r = np.random.RandomState(seed)
    bits = d.itemsize * 8
    x = r.randint(0, 1 << 62, n, dtype=np.uint64) * np.uint64(4) + r.randint(0, 4, n).astype(np.uint64)
    if kind == "runs":  # a few values of the high bits, random low ones: long runs out of order
        hi = r.randint(0, 5, n).astype(np.uint64) << np.uint64(bits - 8)
        x = hi | (x & np.uint64((1 << (bits - 26)) - 1))
    elif kind == "pairs":  # neighbours that agree but for their lowest bits
        x = (r.randint(0, max(n // 2, 1), n).astype(np.uint64) << np.uint64(bits - 16)) | (x & np.uint64(3))
    elif kind == "low":
        x = x & np.uint64(0x1FF)
    elif kind == "equal":
        x = np.full(n, 77, np.uint64)
    if d.kind == "f":  # finite values that keep the pattern's order: integers, exact in the mantissa
        return (x >> np.uint64(64 - 22 if kind == "random" else 0)).astype(np.float64).astype(d)
    return x.astype(f"u{d.itemsize}").view(d)


@pytest.mark.parametrize("kind", ["random", "runs", "pairs", "low", "equal"])
@pytest.mark.parametrize("kdt,vdt", TYPES, ids=lambda t: "none" if t is None else np.dtype(t).name)
def test_block_sort_lengths(handle, kdt, vdt, kind):
    desc = kind == "pairs"
    arrays = [make(kdt, n, kind, 100 + n) for n in LENGTHS]
    offs = np.concatenate([[0], np.cumsum(LENGTHS)]).astype(np.uint64)
    keys = np.concatenate(arrays)
    vals = None if vdt is None else np.arange(keys.size).astype(vdt)
    order = np.concatenate([int(o) + stable_order(a, desc) for a, o in zip(arrays, offs[:-1])])
    want_k, want_v = keys[order], None if vals is None else vals[order]
    say(f"block sort segments {np.dtype(kdt).name} {vdt} {kind}")
    tk, tv = dev(keys), None if vals is None else dev(vals)
    handle.sort_segments(tk, dev(offs), tv, descending=desc)
    assert_bits_equal(host(tk), want_k, "segment keys")
    if vals is not None:
        assert_bits_equal(host(tv), want_v, "segment payloads")
    for i, n in enumerate(LENGTHS):
        say(f"block sort {np.dtype(kdt).name} {vdt} {kind} n={n}")
        lo = int(offs[i])
        tk = dev(keys[lo:lo + n])
        if vals is None:
            handle.sort_keys(tk, descending=desc)
        else:
            tv = dev(vals[lo:lo + n])
            handle.sort_pairs(tk, tv, descending=desc)
            assert_bits_equal(host(tv), want_v[lo:lo + n], f"payloads n={n}")
        assert_bits_equal(host(tk), want_k[lo:lo + n], f"keys n={n}")
