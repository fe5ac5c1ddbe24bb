"""How far ahead of the counts its depths report a render is launched (CPU, the rule alone): a host
thread that is late finds the GPU busy, and one that was late once launches all that is left."""
import numpy as np
import pytest

import illume_amd

LIMIT = 1 << 18


def rule(counts, known, launched, depths, limit=LIMIT):
    c = np.ascontiguousarray(counts, dtype=np.uint32)
    return illume_amd.lib().ilm_debug_depths_to_launch(
        c.ctypes.data_as(illume_amd.C.POINTER(illume_amd.C.c_uint32)), known, launched, depths, limit)


def render(counts, depths, lag=0):
    """The waits of a render whose depths find `counts`: at each, the host knows all but the last
    launched depth (lag 0) or all of them (lag 1). Returns the waits and the depths launched."""
    launched, waits = min(3, depths), 0
    while launched < depths:
        waits += 1
        goal = rule(counts, launched - 1 + lag, launched, depths)
        assert launched <= goal <= depths
        if goal == launched:
            break
        launched = goal
    return waits, launched


@pytest.mark.parametrize("ratio", [0.3, 0.45, 0.6, 0.8, 0.95])
@pytest.mark.parametrize("paths", [LIMIT + 1, 1 << 20, 1 << 23, 1 << 26])
@pytest.mark.parametrize("depths", [4, 16, 45, 256])
def test_depths_that_stay_long_need_no_further_word(ratio, paths, depths):
    counts = (paths * ratio ** np.arange(depths)).astype(np.uint32)
    long = int((counts > LIMIT).sum())       # depths with work for the per-depth kernels
    waits, launched = render(counts, depths)
    assert launched >= min(long, depths)
    assert launched <= max(3, long + 2)      # two launches for nothing, as for a host that is never late
    assert waits <= 3                        # and not one for each depth


def test_slower_and_faster_decay_than_foreseen():
    slow = [1 << 24, 1 << 22] + [int(0.93 ** k * (1 << 22)) for k in range(1, 60)]
    long = sum(c > LIMIT for c in slow)
    waits, launched = render(slow, 61)
    assert long <= launched <= long + 2 and waits < 8
    fast = [1 << 24, 15 << 20, 1 << 20] + [1 << 10] * 42
    waits, launched = render(fast, 45)       # it takes the queue for long and gets none that is
    assert launched == 45 or launched <= rule(fast, 2, 3, 45)


def test_late_host_launches_the_rest():
    counts = [1 << 24, 1 << 23, 1 << 22, 1 << 21, 1 << 20] + [0] * 40
    assert rule(counts, 3, 3, 45) == 45
    assert rule(counts, 5, 5, 45) == 45
    assert render([3 << 20, 2 << 20, 1 << 20] + [0] * 42, 45, lag=1) == (1, 45)


def test_short_queues_end_it_and_the_ends_of_the_range_hold():
    assert rule([1 << 20, LIMIT], 2, 3, 45) == 3
    assert rule([1 << 20, 1 << 19, LIMIT], 3, 3, 45) == 3          # late, but nothing is left to launch
    assert rule([1 << 20, LIMIT + 1], 2, 3, 45) == 4
    assert rule([1 << 20, 1 << 20], 2, 3, 45) == 45                # none ends: all of them
    assert rule([1 << 20, 1 << 21], 2, 3, 45) == 45
    assert rule([1 << 20, LIMIT + 1], 2, 3, 3) == 3
    assert rule([0xFFFFFFFF, 0xFFFFFFFE], 2, 3, 256) == 256
    for bad in ((1, 3, 45, LIMIT), (4, 3, 45, LIMIT), (2, 46, 45, LIMIT), (2, 3, 45, 0)):
        assert rule([1 << 20] * 4, *bad) == -1
