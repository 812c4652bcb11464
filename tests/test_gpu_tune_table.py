"""A tuning table set back: shapes that stwo_hip_fft_autotune left on the default
stay on it (the launches are the same ones by name, and the results exact)."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu

# groups that take the matrix passes, a workgroup per column, and butterfly passes
GROUPS = [(16, 70), (10, 16), (15, 2)]
B = 1


@pytest.fixture(scope="module")
def sets():
    out = []
    for n, C in GROUPS:
        evs = [oracle.fill_random(1 << n, 60 + n, c) for c in range(C)]
        tw, itw = oracle.precompute_twiddles(oracle.half_odds_initial(n + B - 1), n + B - 1)
        coeffs = [e.copy() for e in evs]
        oracle.interpolate_columns(coeffs, itw)
        out.append((n, evs, coeffs, oracle.evaluate_polynomials(coeffs, B, tw)))
    return out


def _launches(ctx, sets):
    """Names of the launches of each group's transforms, their results checked."""
    names = []
    for n, evs, coeffs, want in sets:
        tw = ctx.precompute_twiddles(sh.half_odds(n + B - 1))
        cols, outs = [ctx.to_device(e) for e in evs], [ctx.alloc(2 << n) for _ in evs]
        ctx.prof_enable()
        ctx.prof_reset()
        ctx.interpolate_columns(cols, [n] * len(cols), tw)
        ctx.evaluate_polynomials(cols, [n] * len(cols), B, tw, outs)
        names.append(sorted(ctx.prof_read()))
        ctx.prof_enable(False)
        for c, e in zip(cols + outs, coeffs + want):
            assert np.array_equal(c.download(), e)
            c.free()
        tw.destroy()
    return names


def test_default_entries_stay_on_the_default(sets):
    with sh.Context(0) as ctx:
        default = _launches(ctx, sets)
        assert any("mx" in k for k in default[0]) and any("column" in k for k in default[1])
        ctx.fft_tune_set([(n, N, inv, 12, 8, 0) for n, _ in GROUPS for N, inv in ((n, 1), (n + B, 0))])
        assert _launches(ctx, sets) == default
        # another plan stands in the default's place
        ctx.fft_tune_set([(n, N, inv, 12, 5, 9) for n, _ in GROUPS for N, inv in ((n, 1), (n + B, 0))])
        assert not any("mx" in k or "column" in k for names in _launches(ctx, sets) for k in names)
        ctx.fft_tune_clear()
        assert _launches(ctx, sets) == default


def test_report_set_back(sets):
    logs = [n for n, C in GROUPS for _ in range(C)]
    with sh.Context(0) as ctx, sh.Context(0) as other:
        tw = ctx.precompute_twiddles(sh.half_odds(max(logs) + B - 1))
        report = ctx.fft_autotune(logs, B, tw)
        other.fft_tune_set([r[:6] for r in report])
        assert _launches(other, sets) == _launches(ctx, sets)
        tw.destroy()


def test_choices_leave_shared_launches_alone(sets):
    """A plan over all the groups: another choice for each shape moves none out of the
    launches that they share."""
    logs = [n for n, C in GROUPS for _ in range(C)]
    evs = [e for _, es, _, _ in sets for e in es]
    want = [w for _, _, _, ws in sets for w in ws]
    with sh.Context(0) as ctx:
        tw = ctx.precompute_twiddles(sh.half_odds(max(logs) + B - 1))
        cols, outs = [ctx.alloc(1 << n) for n in logs], [ctx.alloc(2 << n) for n in logs]
        layers = ctx.alloc(sh.tree_words(max(logs) + B))
        names = []
        for t0, smax, wg in ((12, 8, 0), (12, 5, 9)):
            ctx.fft_tune_set([(n, N, inv, t0, smax, wg) for n, _ in GROUPS for N, inv in ((n, 1), (n + B, 0))])
            plan = ctx.batch_create(cols, logs, B, tw, outs, layers, use_graph=False)
            for c, e in zip(cols, evs):
                c.upload(e)
            ctx.prof_enable()
            ctx.prof_reset()
            plan.run()
            names.append({k for k in ctx.prof_read() if "mx" in k or "column" in k})
            ctx.prof_enable(False)
            for o, w in zip(outs, want):
                assert np.array_equal(o.download(), w)
            plan.destroy()
        assert names[0] == names[1] and any("mx" in k for k in names[0]) and any("column" in k for k in names[0])
        tw.destroy()
