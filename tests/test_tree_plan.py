"""CPU checks of the one-launch trees through stwo_hip_debug_tree_plan (which
launches nothing): for every run of layers the library accepts -- node layers
and layers with columns, ending at the root or at the next layer with columns,
on a context or in a plan of any height, and FRI layers alone and side by side
-- every level is hashed once, and the counters on which the workgroups of a
launch meet lie within those that there are."""
import ctypes
import os

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "stwo-metal_amd", "libstwo_hip.so")


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(LIB)


def steps(lib, what, top, stop, n, plan):
    out, k = (ctypes.c_uint32 * 48)(), ctypes.c_uint32()
    assert lib.stwo_hip_debug_tree_plan(what, top, stop, n, plan, out, 8, ctypes.byref(k)) == 0
    return [tuple(out[6 * i: 6 * i + 6]) for i in range(k.value)]


def words_met(own, stop):
    """The largest index of a counter on which a launch's workgroups meet, plus one:
    workgroup b of level l counts itself on word base + (b >> s), s the stage's share of
    the levels (at most 8), base past the words of the stages before."""
    base, l = 0, own
    while l > stop:
        stages = -(-(l - stop) // 8)
        s = -(-(l - stop) // stages)
        base += 1 << (l - s)
        l -= s
    return base


def check(lib, what, top, stop, n, plan):
    at = top if what == 0 else top + 1  # the level above the next one to hash
    for first, own, end, wgs, need, there in steps(lib, what, top, stop, n, plan):
        case = (what, top, stop, n, plan, first, own, end)
        assert first == at - 1 and stop <= end <= own <= first, case
        # a workgroup's digests fit its 256 lanes, four each at most
        assert wgs << (10 if first >= 10 else first) >= 1 << first, case
        assert need == words_met(own, end) <= there, case
        assert there <= 1 << 13, case
        at = end
    assert at == stop, (what, top, stop, n, plan)


@pytest.mark.parametrize("top", range(1, 31))
def test_counters_cover_every_run(lib, top):
    for plan in [0] + list(range(top, 31)):
        for stop in range(top):
            check(lib, 0, top, stop, 0, plan)
        for stop in range(top + 1):
            for n in (1, 17):
                check(lib, 1, top, stop, n, plan)


def test_counters_cover_every_fri_layer(lib):
    for column in range(3, 29):
        for lg in range(2, column + 1):
            for jobs in range(1, 17):
                check(lib, 2, lg, 0, jobs, column)
                check(lib, 2, lg, 0, jobs, 0)


def test_only_runs_past_the_counters_are_split(lib):
    """Trees that end at the root, and every run below 2^26, are one launch."""
    for top in range(1, 31):
        assert len(steps(lib, 0, top, 0, 0, 0)) == 1 and len(steps(lib, 0, top, 0, 0, top)) == 1
        for stop in range(top):
            split = len(steps(lib, 0, top, stop, 0, 0)) > 1
            assert not split or (top >= 26 and 14 <= stop < top - 11 or top >= 29), (top, stop)
    assert len(steps(lib, 0, 26, 14, 0, 0)) == 2


def test_bad_arguments(lib):
    out, k = (ctypes.c_uint32 * 48)(), ctypes.c_uint32()
    for what, top, stop, n, plan in [(3, 8, 0, 1, 0), (0, 31, 0, 0, 0), (0, 8, 9, 0, 0), (2, 8, 0, 17, 0), (2, 8, 1, 1, 0)]:
        assert lib.stwo_hip_debug_tree_plan(what, top, stop, n, plan, out, 8, ctypes.byref(k)) == -1
