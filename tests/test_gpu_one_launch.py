"""Merkle trees and FRI layers in one launch, and a group's FRI commits side by
side, against the oracle, bit-exact: tree sizes at the edges of a workgroup's
first digests (64, 256, 1,024) and of the stages above them, trees whose columns
join at lower levels, fold steps of every kind into the layers and into the
single-workgroup tail, last layers on both sides of the size held in the state
(2^6), and the server's jobs of mixed sizes from columns of several alignments
and allocations."""
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


def _tree(ctx, logs, kind, mode):
    top = max(logs)
    cols = [oracle.fill_random(1 << n, 900 + n, i) for i, n in enumerate(logs)]
    bufs = [ctx.to_device(c) for c in cols]
    layers = ctx.zeros(((2 << top) - 1) * 8)
    for _ in range(2):  # the counters are back at zero after a tree
        if kind == "mixed":
            ctx.merkle_commit(bufs, logs, layers, mode)
        else:
            ctx.lifted_commit(bufs, logs, top, layers, mode)
        got = layers.download(((2 << top) - 1) * 8)
        want = (oracle.merkle_commit(cols, mode == sh.HASH_BLAKE2S_M31) if kind == "mixed"
                else oracle.lifted_commit(cols, top, mode == sh.HASH_BLAKE2S_M31))
        assert np.array_equal(got, want)


@pytest.mark.parametrize("lg", [4, 5, 6, 7, 8, 13, 14, 15, 17, 18, 19, 21])
@pytest.mark.parametrize("mode", [sh.HASH_BLAKE2S, sh.HASH_BLAKE2S_M31])
def test_tree_sizes(ctx, lg, mode):
    _tree(ctx, [lg] * 3, "mixed", mode)
    _tree(ctx, [lg] * 2, "lifted", mode)


@pytest.mark.parametrize("logs", [[14, 6], [15, 14, 7, 7], [18, 10, 4], [19, 18, 9], [20, 8, 5], [9, 8, 7, 6, 5, 4]])
def test_trees_joined_below(ctx, logs):
    _tree(ctx, logs, "mixed", sh.HASH_BLAKE2S)
    _tree(ctx, logs, "mixed", sh.HASH_BLAKE2S_M31)


def _evals(n, b, n_cols=4):
    """(columns, their evaluations on the blown-up domain)."""
    L = n + b
    tw, itw = oracle.precompute_twiddles(oracle.half_odds_initial(L - 1), L - 1)
    cols = [oracle.fill_random(1 << n, 500 + n, c) for c in range(n_cols)]
    co = [c.copy() for c in cols]
    oracle.interpolate_columns(co, itw)
    outs = oracle.evaluate_polynomials(co, b, tw)
    return cols, outs


# (trace log, blowup, last layer bound, fold step): the tail entered by the
# circle fold (L = 9), by line folds of 1 to 4 steps, or never; last layers of
# 2^6 and 2^7; a first layer above the 1,024-digest workgroups' line
FRI = [(4, 1, 1, 1), (8, 1, 0, 1), (8, 1, 0, 4), (9, 1, 1, 2), (10, 2, 4, 3), (9, 2, 0, 4), (9, 3, 4, 2), (7, 2, 4, 1),
       (14, 1, 0, 3), (15, 3, 1, 1), (17, 1, 2, 4), (18, 1, 0, 1)]


@pytest.mark.parametrize("n,b,bound,step", FRI)
def test_fri(ctx, n, b, bound, step):
    L = n + b
    _, outs = _evals(n, b)
    tw = ctx.precompute_twiddles(sh.half_odds(L - 1))
    bufs = [ctx.to_device(o) for o in outs]
    for _ in range(2):
        ch = oracle.Channel()
        roots, last, digest, draws = ctx.fri_commit(ch.digest_bytes(), ch.n_draws, sh.FriConfig(b, bound, 3, step),
                                                    bufs, L, tw)
        want_roots, want_last, _ = oracle.fri_commit(ch, oracle.FriConfig(b, bound, 3, step), outs, L)
        assert np.array_equal(np.array(roots), want_roots) and np.array_equal(np.array(last), want_last)
        assert digest == ch.digest_bytes() and draws == ch.n_draws


def test_jobs_side_by_side(ctx):
    """20 jobs in one group (the layer launches take 16), sizes and steps mixed."""
    jobs = []
    for i in range(20):
        n, b, bound, step = FRI[i % len(FRI)]
        jobs.append((min(n, 13), b, bound, step, 4 + i % 3, i % 5))
    keep, ids, want = [], [], []
    with sh.Server(0, 1 << 30, 17, 1, max_group=20) as srv:
        srv.hold(True)
        for n, b, bound, step, n_cols, shift in jobs:
            L = n + b
            cols, outs = _evals(n, b, n_cols)
            root = oracle.lifted_commit(outs, L)[:8]
            ch = oracle.Channel()
            ch.mix_root(root)
            roots, last, _ = oracle.fri_commit(ch, oracle.FriConfig(b, bound, 3, step), outs[:4], L)
            want.append((root, roots, last, ch.digest_bytes()))
            # columns `shift` words off 16-byte alignment, in an allocation per job
            pitch = (1 << n) + 8
            t = ctx.alloc(n_cols * pitch)
            for k, c in enumerate(cols):
                t.upload(c, k * pitch + shift)
            at = [t.at(k * pitch + shift) for k in range(n_cols)]
            keep.append(t)
            ctx.sync()
            ids.append(srv.submit(n_cols, n, b, 0, sh.FriConfig(b, bound, 3, step), cols=at))
        srv.hold(False)
        res = [srv.wait(i) for i in ids]
    for r, (root, roots, last, digest), job in zip(res, want, jobs):
        assert r.status == 0 and r.group_size == 20, job
        assert list(r.trace_root) == list(root), job
        assert r.n_fri_roots == len(roots) and list(r.fri_roots[:8 * len(roots)]) == list(roots.ravel()), job
        assert list(r.last_layer_poly[:last.size]) == list(last.ravel()), job
        assert bytes(r.final_digest) == digest, job


# Leaf layers of full blocks of 16 columns: at the layer's own size or above it in
# one block or several, a remainder after them, tables among the arguments (up to 64
# columns) and in memory, layers that load a block ahead (2^15) and not (2^17)
FULL = [[17] * 16, [15] * 33, [17] * 64, [17] * 65, [15] * 96, [12] * 3 + [15] * 14 + [17] * 20, [9] * 16 + [16] * 17,
        [5] * 30 + [16] * 18 + [17] * 32]


@pytest.mark.parametrize("logs", FULL, ids=["%dx%d" % (len(f), max(f)) for f in FULL])
def test_full_blocks(ctx, logs):
    for mode in (sh.HASH_BLAKE2S, sh.HASH_BLAKE2S_M31):
        _tree(ctx, logs, "mixed", mode)
        _tree(ctx, logs, "lifted", mode)


def test_full_blocks_side_by_side(ctx):
    """The same of several trees in one launch: jobs of one group."""
    jobs, ids, want = [(14, 33), (14, 16), (15, 40), (15, 17)], [], []
    with sh.Server(0, 1 << 30, 17, 1, max_group=len(jobs)) as srv:
        srv.hold(True)
        for n, n_cols in jobs:
            cols, outs = _evals(n, 1, n_cols)
            want.append(oracle.lifted_commit(outs, n + 1)[:8])
            bufs = [ctx.to_device(c) for c in cols]
            ctx.sync()
            ids.append((srv.submit(n_cols, n, 1, 0, sh.FriConfig(1, 1, 3, 1), cols=bufs), bufs))
        srv.hold(False)
        for (i, _), root, job in zip(ids, want, jobs):
            r = srv.wait(i)
            assert r.status == 0 and list(r.trace_root) == list(root), job
