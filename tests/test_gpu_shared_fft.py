"""interpolate_columns, evaluate_polynomials and extend_evals over columns of
several sizes, whose groups share launches, against the oracle, bit-exact: sizes
on both sides of every pass split, the sizes below 2^4 that keep their own
launches, few and many schedules in a launch, columns off 16-byte alignment,
groups that together fill the matrix passes, and column lists where one group's
output is another group's input (then one group after the other, smallest
first)."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu

LISTS = [[4, 5], [1, 2, 3, 4, 5, 6], list(range(1, 20)), [12, 13, 17, 20], [18, 18, 9, 4, 9], [16] * 33 + [14] * 40,
         [15] * 20 + [16] * 20 + [17] * 9 + [4], [21, 10]]


@pytest.fixture(scope="module")
def ctx():
    c = sh.Context(0)
    yield c
    c.close()


def _twiddles(ctx, top):
    return ctx.precompute_twiddles(sh.half_odds(top - 1)), oracle.precompute_twiddles(oracle.half_odds_initial(top - 1), top - 1)


def _place(ctx, logs, shift):
    """A buffer with room for the columns, `shift` words off alignment, and their offsets."""
    offs, at = [], shift
    for n in logs:
        offs.append(at)
        at += max(4, 1 << n) + 4
    return ctx.alloc(at), offs


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("logs", LISTS, ids=lambda l: "%dx%d-%d" % (len(l), min(l), max(l)))
def test_sizes_share_launches(ctx, logs, shift):
    evs = [oracle.fill_random(1 << n, 40 + n, i) for i, n in enumerate(logs)]
    for b in (0, 1, 3):
        top = max(logs) + b
        if top > 22:
            continue
        tw, (etw, eitw) = _twiddles(ctx, top)
        buf, offs = _place(ctx, logs, shift)
        out, ooffs = _place(ctx, [n + b for n in logs], shift)
        cols, outs = [buf.at(o) for o in offs], [out.at(o) for o in ooffs]
        coeffs = [e.copy() for e in evs]
        oracle.interpolate_columns(coeffs, eitw)
        want = oracle.evaluate_polynomials(coeffs, b, etw)

        def load():
            for e, o in zip(evs, offs):
                buf.upload(e, o)

        def check(b_, offs_, expect, what):
            for k, (o, e) in enumerate(zip(offs_, expect)):
                assert np.array_equal(b_.download(len(e), o), e), (what, b, k, logs[k])

        load()
        ctx.interpolate_columns(cols, logs, tw)
        check(buf, offs, coeffs, "interpolate")
        ctx.evaluate_polynomials(cols, logs, b, tw, outs)
        check(out, ooffs, want, "evaluate")
        load()
        ctx.extend_evals(cols, logs, b, tw, outs, True)
        check(out, ooffs, want, "extend")
        check(buf, offs, coeffs, "extend's coefficients")
        buf.free()
        out.free()
        tw.destroy()


def test_groups_that_meet(ctx):
    """Evaluating the columns of 2^6 writes the coefficients of a column of 2^9."""
    tw, (etw, _) = _twiddles(ctx, 10)
    small, big = oracle.fill_random(1 << 6, 3, 0), oracle.fill_random(1 << 9, 4, 0)
    buf = ctx.alloc((1 << 11) + (1 << 10))
    at_small, at_big, at_out = 0, 1 << 6, 1 << 11
    buf.upload(small, at_small)
    buf.upload(big, at_big)
    ctx.evaluate_polynomials([buf.at(at_big), buf.at(at_small)], [9, 6], 1, tw, [buf.at(at_out), buf.at(at_big)])
    first = oracle.evaluate_polynomials([small], 1, etw)[0]
    then = big.copy()
    then[:1 << 7] = first
    assert np.array_equal(buf.download(1 << 10, at_out), oracle.evaluate_polynomials([then], 1, etw)[0])
    buf.free()
    tw.destroy()
