"""Mixed trees whose runs of node layers end far above the root, at a layer with
columns: there a launch's workgroups meet on the most counters (2^24 down to 2^12:
4,096) or would on more than there are (2^26 down to 2^14: two launches).  Against
one commit_on_layer call per layer, every hash of every layer, from a call and from
a plan."""
import numpy as np
import pytest

import stwo_hip as sh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = sh.Context(0)
    yield c
    c.close()


def _check(ctx, layers, cols, logs):
    """The packed tree against commit_on_layer, from the leaves up."""
    top = max(logs)
    prev, chunk = None, 1 << 26
    for l in range(top, -1, -1):
        out = ctx.alloc(8 << l)
        ctx.commit_on_layer(l, prev, [c for c, n in zip(cols, logs) if n == l], out)
        for at in range(0, 8 << l, chunk):
            n = min(chunk, (8 << l) - at)
            assert np.array_equal(out.download(n, at), layers.download(n, sh.layer_offset(l) + at)), l
        if prev is not None:
            prev.free()
        prev = out
    prev.free()


@pytest.mark.parametrize("logs", [[24, 11], [25, 12, 3], [26, 13]])
def test_commit(ctx, logs):
    cols = []
    for i, n in enumerate(logs):
        cols.append(ctx.alloc(1 << n))
        ctx.fill_random(cols[-1], 1 << n, 11, i)
    layers = ctx.zeros(sh.tree_words(max(logs)))
    for _ in range(2):  # the counters are back at zero after a tree
        ctx.merkle_commit(cols, logs, layers)
    _check(ctx, layers, cols, logs)
    for b in cols + [layers]:
        b.free()


def test_plan(ctx):
    """Columns of 2^25 and 2^12 at blowup 2, and a second tree whose steps share launches."""
    sets, bufs, tw = [], [], ctx.precompute_twiddles(sh.half_odds(25))
    for k, logs in enumerate(([25, 12], [17, 12, 5])):
        cols = [ctx.alloc(1 << n) for n in logs]
        outs = [ctx.alloc(2 << n) for n in logs]
        layers = ctx.zeros(sh.tree_words(max(logs) + 1))
        sets.append((cols, logs, 1, outs, layers, sh.TREE_MIXED, sh.HASH_BLAKE2S))
        bufs += cols + outs + [layers]
    plan = ctx.batch_create_multi(sets, tw)
    for seed in (1, 2):
        for cols, logs, *_ in sets:
            for i, (c, n) in enumerate(zip(cols, logs)):
                ctx.fill_random(c, 1 << n, seed, i)
        plan.run()
        ctx.sync()
    for _, logs, _, outs, layers, _, _ in sets:
        _check(ctx, layers, outs, [n + 1 for n in logs])
    plan.destroy()
    for b in bufs:
        b.free()
    tw.destroy()
