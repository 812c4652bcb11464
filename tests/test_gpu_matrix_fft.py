"""The FFT passes on the matrix cores (groups of at least 3 columns of 2^12
to 2^24 coefficients) against the oracle, bit-exact, at the edges of their
ranges: the low pass alone (n = 12), the first and last size of the 4-layer
and the 8-layer top pass (13, 16, 17, 20), the sizes with a vector pass in
between (21, 24), column counts around the low pass's groups of 4 and past
one workgroup's share, blowups 0 to 4 (the table's last) and 5 (back on the
vector passes), and words at the ends of the field's range."""
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


SHAPES = [(12, 0, 4), (12, 1, 5), (12, 4, 3), (13, 2, 3), (14, 1, 9), (16, 1, 4), (16, 4, 3), (17, 0, 3), (17, 3, 6),
          (18, 5, 3), (19, 1, 37), (20, 1, 7), (21, 1, 3), (22, 0, 3), (24, 0, 3)]


def _columns(n, C):
    evs = [oracle.fill_random(1 << n, 70 + n, c) for c in range(C)]
    evs[0][:] = oracle.P - 1
    evs[1][::2] = 0
    evs[1][1::2] = oracle.P - 1
    return evs


@pytest.mark.parametrize("n,b,C", SHAPES)
def test_transforms_vs_oracle(ctx, n, b, C):
    N = n + b
    print("matrix passes n=%d b=%d cols=%d" % (n, b, C), flush=True)
    tw = ctx.precompute_twiddles(sh.half_odds(N - 1))
    etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(N - 1), N - 1)
    evs = _columns(n, C)
    coeffs = [e.copy() for e in evs]
    oracle.interpolate_columns(coeffs, eitw)
    want = oracle.evaluate_polynomials(coeffs, b, etw)
    cols = [ctx.to_device(e) for e in evs]
    outs = [ctx.alloc(1 << N) for _ in range(C)]
    ctx.interpolate_columns(cols, [n] * C, tw)
    for c, w in zip(cols, coeffs):
        assert np.array_equal(c.download(), w)
    ctx.evaluate_polynomials(cols, [n] * C, b, tw, outs)
    for o, w in zip(outs, want):
        assert np.array_equal(o.download(), w)
    for store in (True, False):
        for c, e, o in zip(cols, evs, outs):
            c.upload(e)
            o.upload(np.zeros(1 << N, np.uint32))
        ctx.extend_evals(cols, [n] * C, b, tw, outs, store_coeffs=store)
        for o, w in zip(outs, want):
            assert np.array_equal(o.download(), w)
        if store:
            for c, w in zip(cols, coeffs):
                assert np.array_equal(c.download(), w)
    for x in cols + outs:
        x.free()
    tw.destroy()
