"""The sizes with a pass between the matrix passes (2^21 to 2^24) in groups of few
columns, on both sides of the lines below which those stay on the vector passes (seen
in the launches' names), at blowups 1 to 4, against the oracle."""
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


@pytest.mark.parametrize("n,b,C,matrix", [(21, 2, 3, True), (22, 1, 3, False), (22, 2, 4, True), (23, 0, 3, False),
                                          (23, 1, 4, True), (23, 0, 5, True), (24, 0, 4, True), (24, 0, 5, False),
                                          (24, 0, 6, True)])
def test_few_large_columns(ctx, n, b, C, matrix):
    N = n + b
    tw = ctx.precompute_twiddles(sh.half_odds(N - 1))
    etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(N - 1), N - 1)
    evs = [oracle.fill_random(1 << n, 20 + n, c) for c in range(C)]
    coeffs = [e.copy() for e in evs]
    oracle.interpolate_columns(coeffs, eitw)
    want = oracle.evaluate_polynomials(coeffs, b, etw)
    cols, outs = [ctx.to_device(e) for e in evs], [ctx.alloc(1 << N) for _ in evs]
    ctx.prof_enable()
    ctx.prof_reset()
    ctx.interpolate_columns(cols, [n] * C, tw)
    ctx.evaluate_polynomials(cols, [n] * C, b, tw, outs)
    names = ctx.prof_read()
    ctx.prof_enable(False)
    assert any("mx" in k for k in names) == matrix, names
    for c, w in zip(cols + outs, coeffs + want):
        assert np.array_equal(c.download(), w)
    for c, e in zip(cols, evs):
        c.upload(e)
    ctx.extend_evals(cols, [n] * C, b, tw, outs)
    for o, w in zip(outs, want):
        assert np.array_equal(o.download(), w)
    for x in cols + outs:
        x.free()
    tw.destroy()
