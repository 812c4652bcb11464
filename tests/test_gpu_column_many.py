"""Many small columns at large blowups, on both sides of the line at which they leave
the workgroup-per-column launch (seen in the launches' names), against the oracle."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = sh.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,b,C,column", [(4, 8, 4096, True), (4, 8, 4097, False), (4, 3, 65535, True),
                                          (4, 5, 16384, True), (4, 5, 16385, False), (5, 8, 8192, True), (5, 7, 8193, False),
                                          (6, 5, 16384, True), (6, 5, 16385, False)])
def test_line(ctx, n, b, C, column):
    N, distinct = n + b, 96
    tw = ctx.precompute_twiddles(sh.half_odds(N - 1))
    etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(N - 1), N - 1)
    evs = [oracle.fill_random(1 << n, 50 + n, c) for c in range(distinct)]
    coeffs = [e.copy() for e in evs]
    oracle.interpolate_columns(coeffs, eitw)
    want = np.array(oracle.evaluate_polynomials(coeffs, b, etw))
    pick = np.arange(C) % distinct
    buf, out = ctx.alloc(C << n), ctx.alloc(C << N)
    cols, outs = [buf.at(c << n) for c in range(C)], [out.at(c << N) for c in range(C)]
    for what, start in (("evaluate", coeffs), ("extend", evs)):
        buf.upload(np.array(start)[pick].ravel())
        ctx.prof_enable()
        ctx.prof_reset()
        if what == "evaluate":
            ctx.evaluate_polynomials(cols, [n] * C, b, tw, outs)
        else:
            ctx.extend_evals(cols, [n] * C, b, tw, outs)
        names = ctx.prof_read()
        ctx.prof_enable(False)
        assert any("column" in k for k in names) == column, names
        got = out.download().reshape(C, -1)
        for k in range(distinct):
            assert np.all(got[k::distinct] == want[k]), (what, k)
    buf.free()
    out.free()
    tw.destroy()
