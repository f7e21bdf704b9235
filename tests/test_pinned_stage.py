"""The places that the small transfers of a call take in the pinned buffer: blocks
read together never share bytes, wherever the hand-out starts over (CPU, the
library's own header against plain memory)."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

SOURCE = Path(__file__).resolve().parent / "cpp" / "stage_test.cpp"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("stage") / "stage_test"
    subprocess.run(["g++", "-O1", "-Wall", "-Wextra", "-Werror", "-std=c++17", str(SOURCE), "-o", str(out)], check=True)
    return out


@pytest.mark.parametrize("capacity,rounds,seed", [(4096, 3000, 1), (4096 + 17, 3000, 2), (65536, 500, 3)])
def test_blocks_read_together_come_back_whole(program, capacity, rounds, seed):
    r = subprocess.run([str(program), str(capacity), str(rounds), str(seed)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
