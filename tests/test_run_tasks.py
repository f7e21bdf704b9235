"""Forward progress of the runs that workgroups share (CPU model, no GPU):
workgroups take tasks by one ticket, phase after phase, and a task waits until the
phase before its own is done (gpusort_amd/csrc/radix_ties.h, long_run_kernel).
Whatever number of workgroups is resident, and in whatever order they get on,
every task is run, none before its phase may start."""
from __future__ import annotations

import random

import pytest


def phase_sizes(tasks: int, runs: int, digits: int) -> list[int]:
    return [tasks] + [tasks, runs, tasks] * digits + [tasks]


def place(ticket: int, tasks: int, runs: int, digits: int):
    """Phase and place in it of a ticket, by the kernel's arithmetic; None past the end."""
    at = ticket
    if at < tasks:
        return 0, at
    at -= tasks
    per = 2 * tasks + runs
    turn = min(at // per, digits)
    at -= turn * per
    phase = 1 + 3 * turn
    if turn == digits:
        return (phase, at) if at < tasks else None
    if at >= tasks + runs:
        return phase + 2, at - tasks - runs
    if at >= tasks:
        return phase + 1, at - tasks
    return phase, at


@pytest.mark.parametrize("tasks,runs,digits", [(4, 1, 1), (5, 2, 4), (37, 3, 7), (4, 1, 0)])
def test_tickets_are_every_task_once_in_phase_order(tasks, runs, digits):
    sizes = phase_sizes(tasks, runs, digits)
    want = [(p, i) for p, n in enumerate(sizes) for i in range(n)]
    assert [place(t, tasks, runs, digits) for t in range(len(want))] == want
    assert place(len(want), tasks, runs, digits) is None
    assert len(sizes) <= 24  # the control block's counters


@pytest.mark.parametrize("resident", [1, 2, 17, 256])
def test_every_task_runs(resident):
    tasks, runs, digits = 37, 3, 7
    sizes = phase_sizes(tasks, runs, digits)
    rng = random.Random(resident)
    done = [0] * len(sizes)
    ticket, held, steps = 0, [], 0
    while sum(done) < sum(sizes):
        while len(held) < resident and ticket < sum(sizes):  # a free workgroup takes the next ticket
            held.append(place(ticket, tasks, runs, digits)[0])
            ticket += 1
        ready = [i for i, p in enumerate(held) if p == 0 or done[p - 1] == sizes[p - 1]]
        assert ready, "every resident workgroup waits"
        done[held.pop(rng.choice(ready))] += 1
        steps += 1
    assert done == sizes and steps == sum(sizes)
