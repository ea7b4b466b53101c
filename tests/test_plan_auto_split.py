"""The automatic split of a type-1 work plan: with few records in reach, heavy
blocks are cut into parts of an even share over 2048 waves.  A batch sizes its
partial-sum scratch before any kernel runs, so a plan's heavy parts may never
exceed that bound.  The engine's own split rule, part length and bound
(tile_index.hpp, shared by the planning kernel and the batch's host code) run
on the CPU over random and lopsided block totals; a bound of too few waves
(planted here) must be exceeded.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

REPLAY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "replay")


@pytest.fixture(scope="module")
def plan_lib():
    subprocess.run(["make", "-s", "-C", REPLAY], check=True)
    L = ctypes.CDLL(os.path.join(REPLAY, "_build", "libtile_replay.so"))
    L.replay_plan.restype = ctypes.c_int64
    L.replay_plan.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_uint32, ctypes.c_uint32,
                              ctypes.c_int, ctypes.c_int64, ctypes.c_double, ctypes.c_int64,
                              ctypes.c_void_p]
    return L


def _plan(L, totals, capacity, auto=True, light=0, min_part=0):
    """(items, heavy parts, heavy blocks, records per part), slots: every
    record in reach of one block."""
    t = np.ascontiguousarray(totals, dtype=np.uint32)
    out = np.zeros(4, dtype=np.uint32)
    slots = L.replay_plan(t.ctypes.data, t.size, light, min_part, int(auto), capacity, 1.0,
                          int(t.sum(dtype=np.int64)), out.ctypes.data)
    assert slots >= 0
    return out.tolist(), slots


def _sets():
    rng = np.random.default_rng(5)
    yield np.full(256, 740)
    yield np.full(1, 5_000_000)
    yield np.full(1, 300)
    yield np.array([1_000_000] + [1] * 4000)
    for blocks in (1, 7, 100, 3000, 40000):
        for scale in (10, 300, 2000, 60000):
            yield rng.integers(0, 2 * scale, blocks)
            yield (rng.pareto(1.0, blocks) * scale).astype(np.int64).clip(0, 1 << 31)


@pytest.mark.parametrize("light,min_part", [(0, 0), (300, 1), (1 << 20, 1 << 16)])
@pytest.mark.parametrize("auto", [True, False])
@pytest.mark.parametrize("capacity", [64, 4096, 131072])
def test_parts_fit_the_batch_bound(plan_lib, capacity, auto, light, min_part):
    for totals in _sets():
        (items, parts, heavy, _), slots = _plan(plan_lib, totals, capacity, auto, light,
                                                min_part)
        assert parts <= slots <= capacity
        assert items == totals.size - heavy + parts


def test_small_sets_are_split_over_the_chip(plan_lib):
    """256 tiles of 740 records: parts of at least 128, up to one a wave; a
    plan with a caller's own values keeps them."""
    (items, parts, heavy, length), _ = _plan(plan_lib, np.full(256, 740), 131072)
    assert heavy == 256 and length == 128 and items == parts == 256 * 6
    (items, parts, _, _), _ = _plan(plan_lib, np.full(256, 740), 131072, auto=False)
    assert items == 256 and parts == 0
    # large sets: the automatic split changes nothing
    for totals in (np.full(20000, 4000), np.full(3000, 60000)):
        assert _plan(plan_lib, totals, 131072) == _plan(plan_lib, totals, 131072, auto=False)


def test_planted_small_bound_is_exceeded(plan_lib):
    """The sets above reach the bound: with an eighth of its waves the parts
    of some would not fit."""
    assert any(_plan(plan_lib, t, 131072)[0][1] > t.size + max(2 * int(t.sum()) // 1024, 2048 // 8)
               for t in _sets())
