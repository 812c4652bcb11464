"""eval_at_point where a workgroup takes more blocks of 2^11 coefficients than it holds
factors for (64), and where there are more runs of equal-sized columns than counters
(8,192; then a workgroup a run), against the oracle.  The columns repeat few buffers."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu

POINT = ([5, 1 << 30, 77, 123456789], [2147483646, 3, 999, 31])


@pytest.fixture(scope="module")
def ctx():
    c = sh.Context(0)
    yield c
    c.close()


def _columns(ctx, logs):
    """A buffer of each log size, its coefficients' value at POINT by the oracle."""
    out = {}
    for n in set(logs):
        c = oracle.fill_random(1 << n, 13, n)
        c[: 1 << 4] = oracle.P - 1
        out[n] = (ctx.to_device(c), oracle.eval_at_point(c, POINT))
    return out


@pytest.mark.parametrize("logs", [[24] * 56, [24] * 50 + [23] * 7 + [12] * 3], ids=["7 runs", "mixed"])
def test_many_blocks_a_workgroup(ctx, logs):
    cols = _columns(ctx, logs)
    got = ctx.eval_at_point([cols[n][0] for n in logs], logs, POINT)
    for k, n in enumerate(logs):
        assert tuple(int(w) for w in got[k]) == tuple(int(w) for w in cols[n][1]), k
    for b, _ in cols.values():
        b.free()


def test_more_runs_than_counters(ctx):
    logs = [12, 13] * 4100
    cols = _columns(ctx, logs)
    got = ctx.eval_at_point([cols[n][0] for n in logs], logs, POINT)
    assert np.array_equal(got, np.array([[int(w) for w in cols[n][1]] for n in logs], dtype=np.uint32))
    for b, _ in cols.values():
        b.free()
