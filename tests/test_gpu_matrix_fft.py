"""The FFT passes on the matrix cores (groups of at least 3 columns with a
low-pass unit, 4 columns x 2^12 words, for every CU) against the oracle,
bit-exact, at the edges of their ranges: the low pass alone (n = 12), the
first and last size of the 4-layer and the 8-layer top pass (13, 16, 17, 20),
the sizes with a vector pass in between (21, 24), column counts off the low
pass's groups of 4, blowups 0 to 2 (the table's last) and 3 (back on the vector
passes), words at the ends of the field's range, and one batched plan of
several such groups."""
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


SHAPES = [(12, 0, 1021), (12, 2, 1023), (13, 1, 510), (14, 1, 255), (16, 2, 61), (16, 3, 61), (17, 0, 29), (18, 1, 18),
          (19, 2, 9), (20, 1, 3), (20, 2, 5), (21, 1, 3), (22, 0, 3), (24, 0, 3)]


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


def test_batched_groups_vs_oracle(ctx):
    """One plan over groups that share the matrix launches (at least 32 units
    each) and groups that stay on the vector passes."""
    logs = [11] * 5 + [12] * 130 + [13] * 70 + [15] * 35 + [16] * 2 + [17] * 6 + [20] * 3
    b = 1
    top = max(logs) + b
    tw = ctx.precompute_twiddles(sh.half_odds(top - 1))
    etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(top - 1), top - 1)
    evs = [oracle.fill_random(1 << lg, 17, i) for i, lg in enumerate(logs)]
    coeffs = [e.copy() for e in evs]
    oracle.interpolate_columns(coeffs, eitw)
    want = oracle.evaluate_polynomials(coeffs, b, etw)
    root = oracle.merkle_commit(want)[:8]
    cols = [ctx.to_device(e) for e in evs]
    outs = [ctx.alloc(1 << (lg + b)) for lg in logs]
    layers = ctx.alloc(sh.tree_words(top))
    plan = ctx.batch_create(cols, logs, b, tw, outs, layers)
    for _ in range(2):
        for c, e in zip(cols, evs):
            c.upload(e)
        plan.run()
        for c, w in zip(cols, coeffs):
            assert np.array_equal(c.download(), w)
        for o, w in zip(outs, want):
            assert np.array_equal(o.download(), w)
        assert np.array_equal(layers.download(8), root)
    plan.destroy()
    for x in cols + outs + [layers]:
        x.free()
    tw.destroy()
