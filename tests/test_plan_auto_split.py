"""The automatic split of a type-1 work plan (spread.hip plan_blocks): with
few records in reach, heavy blocks are cut into parts of an even share over
2048 waves.  A batch sizes its partial-sum scratch from blocks + max(2 reach
M / smallest part, 2048) before any kernel runs (plan.hip,
execute_type1_many_t), so the parts may never exceed that.  Replayed on the
CPU over random and lopsided block totals; a share rounded down (planted)
must break the bound.
"""
import numpy as np
import pytest

WAVES, FLOOR = 2048, 128


def _parts(totals, capacity, round_up=True, light=4096, min_part=1024):
    total = int(totals.sum())
    share = -(-total // WAVES) if round_up else total // (4 * WAVES)
    part = max(share, FLOOR if round_up else 1)
    if 2 * part < light:
        light, min_part = 2 * part, min(part, min_part)
    while 2 * int((totals > light).sum()) > capacity and light < 0x7FFFFFFF:
        light *= 2
    heavy = totals[totals > light]
    spare = capacity - heavy.size if capacity > heavy.size else 1
    length = max(-(-int(heavy.sum()) // spare), min_part)
    n = -(-heavy // length)
    return int(n[n > 1].sum())


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


@pytest.mark.parametrize("capacity", [64, 4096, 131072])
def test_automatic_parts_fit_the_batch_bound(capacity):
    for totals in _sets():
        bound = min(capacity, totals.size + max(2 * int(totals.sum()) // 1024, WAVES))
        assert _parts(totals, capacity) <= bound


def test_planted_small_share_is_caught():
    assert any(_parts(t, 131072, round_up=False) > t.size + max(2 * int(t.sum()) // 1024, WAVES)
               for t in _sets())
