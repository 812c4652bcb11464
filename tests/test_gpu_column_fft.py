"""Small columns, a workgroup each, against the oracle, bit-exact: every size of
the path at every blowup up to the first domain above it (2^14), odd and even
numbers of layers, words at the ends of the field's range, coefficients kept and
dropped, the first column count that leaves the path, and one plan whose sets
take it in each direction."""
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


def _columns(n, C):
    evs = [oracle.fill_random(1 << n, 80 + n, c) for c in range(C)]
    evs[0][:] = oracle.P - 1
    evs[1][::2] = 0
    evs[1][1::2] = oracle.P - 1
    return evs


@pytest.mark.parametrize("n,C", [(n, 3) for n in range(4, 14)] + [(12, 512), (12, 513), (4, 700)])
def test_columns(ctx, n, C):
    evs = _columns(n, C)
    for b in range(0, 15 - n if n > 10 else 4):
        N = n + b
        tw = ctx.precompute_twiddles(sh.half_odds(N - 1))
        etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(N - 1), N - 1)
        coeffs = [e.copy() for e in evs]
        oracle.interpolate_columns(coeffs, eitw)
        want = np.concatenate(oracle.evaluate_polynomials(coeffs, b, etw))
        buf, out = ctx.alloc(C << n), ctx.alloc(C << N)
        cols, outs = [buf.at(k << n) for k in range(C)], [out.at(k << N) for k in range(C)]
        for store in (False, True):
            buf.upload(np.concatenate(evs))
            out.upload(np.zeros(C << N, dtype=np.uint32))
            ctx.extend_evals(cols, [n] * C, b, tw, outs, store)
            assert np.array_equal(out.download(), want), ("extend", b, store)
        assert np.array_equal(buf.download(), np.concatenate(coeffs)), ("coefficients", b)
        out.upload(np.zeros(C << N, dtype=np.uint32))
        ctx.evaluate_polynomials(cols, [n] * C, b, tw, outs)
        assert np.array_equal(out.download(), want), ("evaluate", b)
        buf.upload(np.concatenate(evs))
        ctx.interpolate_columns(cols, [n] * C, tw)
        assert np.array_equal(buf.download(), np.concatenate(coeffs)), ("interpolate", b)
        buf.free()
        out.free()
        tw.destroy()


def test_plan_in_each_direction(ctx):
    """Interpolations, evaluations of what they write, and both at once, of mixed small sizes."""
    logs, b = [4, 7, 10, 11, 12], 1
    top = max(logs) + b
    tw = ctx.precompute_twiddles(sh.half_odds(top - 1))
    etw, eitw = oracle.precompute_twiddles(oracle.half_odds_initial(top - 1), top - 1)
    evs = [oracle.fill_random(1 << n, 90 + n, 0) for n in logs]
    coeffs = [e.copy() for e in evs]
    oracle.interpolate_columns(coeffs, eitw)
    want = oracle.evaluate_polynomials(coeffs, b, etw)
    tree = oracle.lifted_commit(want, top)
    first, both = [ctx.to_device(e) for e in evs], [ctx.to_device(e) for e in evs]
    outs = [[ctx.alloc(1 << (n + b)) for n in logs] for _ in range(2)]
    layers = [ctx.alloc(sh.tree_words(top)) for _ in range(2)]
    plan = ctx.batch_create_multi(
        [(first, logs, b, None, None, sh.TREE_LIFTED, sh.HASH_BLAKE2S, sh.BATCH_IFFT),
         (first, logs, b, outs[0], layers[0], sh.TREE_LIFTED, sh.HASH_BLAKE2S, sh.BATCH_RFFT),
         (both, logs, b, outs[1], layers[1], sh.TREE_LIFTED, sh.HASH_BLAKE2S)], tw)
    for _ in range(3):
        for c, d, e in zip(first, both, evs):
            c.upload(e)
            d.upload(e)
        plan.run()
        ctx.sync()
        for c, d, e in zip(first, both, coeffs):
            assert np.array_equal(c.download(), e) and np.array_equal(d.download(), e)
        for k in range(2):
            for o, e in zip(outs[k], want):
                assert np.array_equal(o.download(), e)
            assert np.array_equal(layers[k].download(), tree)
    plan.destroy()
    tw.destroy()
