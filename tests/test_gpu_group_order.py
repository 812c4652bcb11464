"""Column lists of several sizes where one group's words are another's: the groups run
smallest first, also those below 2^4, whose launches are their own, and columns
evaluated in place.  Against the oracle, group by group."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu

TOP = 11
SIZE = 1 << 13


@pytest.fixture(scope="module")
def ctx():
    c = sh.Context(0)
    yield c
    c.close()


# (blowup, [(log size, offset of the column, offset of its evaluations)]), largest
# first as the caller gives them: every input read, then written, by another group
CASES = {
    "small's output in large's input": (1, [(9, 1024, 4096), (6, 128, 512), (2, 0, 1032)]),
    "large's output over small's input": (1, [(9, 4096, 0), (6, 6000, 6400), (2, 100, 7000)]),
    "both among the smallest": (2, [(7, 4096, 2048), (5, 1024, 1200), (3, 64, 4100), (2, 32, 64)]),
    "in place, one column inside another": (0, [(9, 0, 0), (6, 64, 64), (3, 72, 72)]),
    "in place over 2^4 alone": (0, [(9, 1024, 1024), (6, 1088, 1088)]),
}


@pytest.mark.parametrize("case", CASES)
def test_smallest_first(ctx, case):
    b, cols = CASES[case]
    tw = ctx.precompute_twiddles(sh.half_odds(TOP - 1))
    etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(TOP - 1), TOP - 1)
    start = oracle.fill_random(SIZE, 77, 0)
    logs = [n for n, _, _ in cols]

    def interpolate(w, n, at):
        c = [w[at: at + (1 << n)].copy()]
        oracle.interpolate_columns(c, eitw)
        w[at: at + (1 << n)] = c[0]

    def evaluate(w, n, at, to):
        w[to: to + (1 << (n + b))] = oracle.evaluate_polynomials([w[at: at + (1 << n)].copy()], b, etw)[0]

    buf = ctx.alloc(SIZE)
    ins, outs = [buf.at(i) for _, i, _ in cols], [buf.at(o) for _, _, o in cols]
    for what in ("interpolate", "evaluate", "extend"):
        want = start.copy()
        for n, i, o in sorted(cols):
            if what != "evaluate":
                interpolate(want, n, i)
            if what != "interpolate":
                evaluate(want, n, i, o)
        buf.upload(start)
        if what == "interpolate":
            ctx.interpolate_columns(ins, logs, tw)
        elif what == "evaluate":
            ctx.evaluate_polynomials(ins, logs, b, tw, outs)
        else:
            ctx.extend_evals(ins, logs, b, tw, outs, store_coeffs=True)
        assert np.array_equal(buf.download(), want), what
    buf.free()
    tw.destroy()
