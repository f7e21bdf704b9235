"""The gather's scratch gives way: a call that finds no device memory gives back
what an earlier gather on the same handle kept before it fails, and the next gather
takes its scratch anew."""
from __future__ import annotations

import pytest
from gpu_util import say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_a_call_without_memory_gives_back_the_scratch_of_a_gather():
    import gpusort_amd

    n = 1 << 25
    gen = torch.Generator(device="cuda").manual_seed(1)
    idx = torch.randint(0, n, (n,), generator=gen, device="cuda")
    src = torch.randint(0, 255, (n,), generator=gen, device="cuda", dtype=torch.uint8)
    dst = torch.empty_like(src)
    k = torch.randint(0, (1 << 31) - 1, (1 << 20,), generator=gen, device="cuda", dtype=torch.int32)
    h = gpusort_amd.Handle(0)
    try:
        h.gather(src, idx, dst)
        assert torch.equal(dst, src[idx])
        assert h.arena_bytes() > 6 * n, "the gather keeps its scratch"
        # 2^38 keys need a workspace of a terabyte: refused before anything is launched.
        say("sort without memory for its workspace")
        status = h.lib.gs_sort_keys(h.h, gpusort_amd.I32, k.data_ptr(), 1 << 38, 0)
        assert status == 2, h.lib.gs_last_error()
        assert h.arena_bytes() < 6 * n, "the scratch was given back"
        dst.zero_()
        h.gather(src, idx, dst)
        assert torch.equal(dst, src[idx])
    finally:
        h.close()
