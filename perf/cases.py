"""The work that users of this framework have it do, as cases to time.

A case is one pass through public entry points of the binding
(stwo-metal_amd/stwo_hip.py) on buffers that already lie on the device:

  commit     a trace is extended (interpolate + evaluate at the blowup) and
             committed to a Blake2s Merkle tree; with `store` the trace columns
             become coefficients, without it the trace is generated by the same
             pass (wide-Fibonacci rows) and its coefficients are dropped, the
             prover's default
  batch      a batch plan (one graph) over columns of uneven sizes, mixed tree
  prove      a whole wide-Fibonacci prove: trace commit, composition, OODS
             samples, FRI quotients, FRI, proof of work, decommitment
  fri        the FRI commit chain on one secure column
  interp     columns read in natural order, bit reversed and interpolated
  evaluate   stored coefficients evaluated on a larger domain
  open       polynomials sampled at a secure point and the FRI quotients of
             their evaluations at that point
  serve      a burst of commit + FRI jobs through the server

Every output is whole numbers (field elements, hash words, proof bytes), so
the outputs of two builds are equal word for word or wrong: exact() has no
value to give.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stwo-metal_amd"))
import stwo_hip as sh  # noqa: E402

P = sh.P
DEV = "cuda:0"


def listed():
    return [
        # the smallest call: a short public-input or lookup table committed by itself
        dict(name="commit_16x2e10", op="commit", cols=16, lo=10, hi=10, blowup=1, store=True, lifted=False),
        # a small trace at the default blowup
        dict(name="commit_16x2e16", op="commit", cols=16, lo=16, hi=16, blowup=1, store=True, lifted=False),
        # a wide trace of a large program, coefficients dropped (the prover's default)
        dict(name="commit_256x2e20_b4", op="commit", cols=256, lo=20, hi=20, blowup=2, store=False, lifted=False),
        # a zkVM's components: many columns of uneven heights under one root
        dict(name="batch_1024_uneven", op="batch", cols=1024, lo=10, hi=22, blowup=1),
        # the end-to-end benchmark prove
        dict(name="prove_256x2e18", op="prove", cols=256, log=18, store=True),
        # a small proof, where latency counts
        dict(name="prove_40x2e11", op="prove", cols=40, log=11, store=False),
        # FRI of a large proof, last layer 2^4
        dict(name="fri_2e22", op="fri", log=22, blowup=1, last=3, step=1),
        # FRI of a small proof folding three times a layer
        dict(name="fri_2e14_step3", op="fri", log=14, blowup=2, last=0, step=3),
        # columns of uneven heights interpolated from natural order
        dict(name="interp_45_ragged", op="interp", cols=45, lo=9, hi=19),
        # stored coefficients evaluated on the composition domain
        dict(name="evaluate_100x2e17_b2", op="evaluate", cols=100, lo=17, hi=17, blowup=1),
        # OODS samples and FRI quotients of a trace and its composition columns
        dict(name="open_264x2e18", op="open", cols=264, lo=18, hi=18, blowup=1),
        # clients' jobs arriving together
        dict(name="serve_burst", op="serve", jobs=12, cols=96, lo=12, hi=17),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["commit", "commit", "batch", "prove", "fri", "interp", "evaluate", "open", "serve"])
    if op == "commit":
        lo = rng.randint(8, 20)
        hi, store = lo, rng.random() < 0.5
        if store:
            hi = rng.randint(lo, min(20, lo + 3))
        b = rng.randint(1, 2)
        most = max(4, min(300, (1 << 28) >> hi))
        return dict(op=op, cols=_log_int(rng, 4, most), lo=lo, hi=hi, blowup=b, store=store, lifted=rng.random() < 0.5)
    if op == "batch":
        lo = rng.randint(6, 14)
        return dict(op=op, cols=_log_int(rng, 20, 1100), lo=lo, hi=rng.randint(lo + 2, 21), blowup=rng.randint(1, 2))
    if op == "prove":
        return dict(op=op, cols=_log_int(rng, 5, 300), log=rng.randint(6, 18), store=rng.random() < 0.5)
    if op == "fri":
        return dict(op=op, log=rng.randint(9, 22), blowup=rng.randint(1, 3), last=rng.randint(0, 4), step=rng.randint(1, 3))
    if op == "interp":
        lo = rng.randint(4, 18)
        return dict(op=op, cols=_log_int(rng, 2, 80), lo=lo, hi=rng.randint(lo, min(21, lo + 10)))
    if op == "evaluate":
        lo = rng.randint(4, 19)
        return dict(op=op, cols=_log_int(rng, 2, 200), lo=lo, hi=rng.randint(lo, min(20, lo + 2)), blowup=rng.randint(0, 3))
    if op == "open":
        lo = rng.randint(6, 18)
        return dict(op=op, cols=_log_int(rng, 5, 300), lo=lo, hi=rng.randint(lo, min(18, lo + 4)), blowup=rng.randint(1, 2))
    lo = rng.randint(8, 14)
    return dict(op=op, jobs=rng.randint(2, 16), cols=_log_int(rng, 8, 128), lo=lo, hi=rng.randint(lo, 17))


# ---- the program's handles and buffers -----------------------------------------

_shared = []


def _ctx():
    """The program's one context."""
    if not _shared:
        _shared.append(sh.Context(0))
    return _shared[0]


def _close(h):
    """Ends a plan, twiddle tree or server that a dropped state held."""
    (h.close if isinstance(h, sh.Server) else h.destroy)()


class State:
    """What a program keeps between calls; its handles end with it."""

    def __init__(self, **kw):
        self.handles = []
        self.__dict__.update(kw)

    def __del__(self):
        if self.handles and _shared:
            _shared[0].sync()
            for h in self.handles:
                _close(h)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _felts(g, n):
    """n field elements (canonical words) on the device."""
    return torch.randint(0, P, (n,), generator=g, device=DEV, dtype=torch.int32)


def _words(n):
    return torch.zeros(n, device=DEV, dtype=torch.int32)


def _views(buf, logs):
    """Addresses of columns of these log sizes laid one after the other."""
    out, at = [], buf.data_ptr()
    for lg in logs:
        out.append(at)
        at += 4 << lg
    return out


def _logs(case):
    """Column heights: spread over [lo, hi] in a fixed order, the batch's more
    often small (P(lo + j) ~ 0.7^j) with each height's count whole."""
    n, lo, hi = case["cols"], case["lo"], case["hi"]
    if case["op"] == "batch":
        rng = np.random.default_rng(3)
        w = np.array([0.7 ** j for j in range(hi - lo + 1)])
        return [int(lo + j) for j in rng.choice(len(w), size=n, p=w / w.sum())]
    return [lo + (5 * i) % (hi - lo + 1) for i in range(n)]


def _job_list(case):
    """(columns, log size, log blowup) of each job of a burst."""
    out = []
    for k in range(case["jobs"]):
        lg = case["lo"] + (3 * k) % (case["hi"] - case["lo"] + 1)
        out.append((max(4, case["cols"] >> (k % 4)) + k % 3, lg, 1 + k % 2))
    return out


def _padded(a, n):
    """a in the first len(a) places of n zeros."""
    out = np.zeros(n, dtype=a.dtype)
    out[: len(a)] = a
    return out


# QM31 = CM31[u] / (u^2 - 2 - i) on host integers, for one random point.
def _cmul(a, b):
    return ((a[0] * b[0] - a[1] * b[1]) % P, (a[0] * b[1] + a[1] * b[0]) % P)


def _qmul(x, y):
    a, b, c, d = x[:2], x[2:], y[:2], y[2:]
    bd = _cmul(_cmul(b, d), (2, 1))
    ac, ad, bc = _cmul(a, c), _cmul(a, d), _cmul(b, c)
    return tuple((p + q) % P for p, q in zip(ac + ad, bd + bc))


def _qinv(x):
    e, r = P ** 4 - 2, (1, 0, 0, 0)
    while e:
        if e & 1:
            r = _qmul(r, x)
        x = _qmul(x, x)
        e >>= 1
    return r


def _secure_point(rng):
    """((1 - t^2) / (1 + t^2), 2t / (1 + t^2)) for a random t."""
    t = tuple(int(v) for v in rng.integers(0, P, 4))
    t2 = _qmul(t, t)
    one = (1, 0, 0, 0)
    d = _qinv(tuple((a + b) % P for a, b in zip(one, t2)))
    return (_qmul(tuple((a - b) % P for a, b in zip(one, t2)), d), _qmul(tuple(2 * a % P for a in t), d))


def prepare(case, seed):
    ctx, g, op = _ctx(), _gen(seed), case["op"]
    s = State(case=case)

    def twiddles(log_size):
        s.tw = ctx.precompute_twiddles(sh.half_odds(log_size - 1))
        s.handles.append(s.tw)

    if op in ("commit", "batch", "evaluate", "interp"):
        s.logs = _logs(case)
        total = sum(1 << lg for lg in s.logs)
        top = max(s.logs) + case.get("blowup", 0)
        twiddles(top)
        fresh = op == "commit" and not case["store"]
        s.trace = _words(total) if fresh else _felts(g, total)
        s.cols = _views(s.trace, s.logs)
        if fresh:
            s.first = _felts(g, 2 << case["lo"])
        if op != "interp":
            s.out_logs = [lg + case["blowup"] for lg in s.logs]
            s.evals = _words(total << case["blowup"])
            s.outs = _views(s.evals, s.out_logs)
        if op in ("commit", "batch"):
            s.top = top
            s.layers = _words(sh.tree_words(top))
        if op == "batch":
            torch.cuda.synchronize()
            s.plan = ctx.batch_create(s.cols, s.logs, case["blowup"], s.tw, s.outs, s.layers.data_ptr())
            s.handles.insert(0, s.plan)
    elif op == "prove":
        twiddles(case["log"] + 1)
        s.first = _felts(g, 2 << case["log"])
    elif op == "fri":
        lg, deg = case["log"], case["log"] - case["blowup"]
        twiddles(lg)
        coeffs = _felts(g, 4 << deg)
        s.column = _words(4 << lg)
        s.coords = _views(s.column, [lg] * 4)
        torch.cuda.synchronize()
        for c, o in zip(_views(coeffs, [deg] * 4), s.coords):
            ctx.evaluate(c, deg, sh.canonic_domain(lg), s.tw, o)
        ctx.sync()
        s.config = sh.FriConfig(case["blowup"], min(case["last"], deg - 1), 3, case["step"])
        s.digest = bytes(int(v) for v in np.random.default_rng(seed).integers(0, 256, 32))
    elif op == "open":
        b = case["blowup"]
        s.logs = _logs(case)
        s.out_logs = [lg + b for lg in s.logs]
        total = sum(1 << lg for lg in s.logs)
        twiddles(max(s.out_logs))
        s.coeffs = _felts(g, total)
        s.cols = _views(s.coeffs, s.logs)
        s.evals = _words(total << b)
        s.outs = _views(s.evals, s.out_logs)
        s.lifting = max(s.out_logs)
        s.quotients = _words(4 << s.lifting)
        torch.cuda.synchronize()
        ctx.evaluate_polynomials(s.cols, s.logs, b, s.tw, s.outs)
        ctx.sync()
        rng = np.random.default_rng(seed)
        s.point = _secure_point(rng)
        s.alpha = [int(v) for v in rng.integers(0, P, 4)]
    else:
        s.jobs = _job_list(case)
        s.traces = [_felts(g, n << lg) for n, lg, _ in s.jobs]
        torch.cuda.synchronize()
        s.server = sh.Server(0, 4 << 30, case["hi"] + 2, 4)
        s.handles.append(s.server)
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, case = _ctx(), s.case
    op = case["op"]
    if op == "commit":
        if not case["store"]:
            n = case["lo"]
            a = s.first.data_ptr()
            ctx.wide_fib_trace(s.cols, n, a, a + (4 << n))
        ctx.extend_evals(s.cols, s.logs, case["blowup"], s.tw, s.outs, store_coeffs=case["store"])
        if case["lifted"]:
            ctx.lifted_commit(s.outs, s.out_logs, s.top, s.layers.data_ptr())
        else:
            ctx.merkle_commit(s.outs, s.out_logs, s.layers.data_ptr())
        out = {"evals": s.evals, "layers": s.layers}
        if case["store"]:
            out["coeffs"] = s.trace
        return out
    if op == "batch":
        s.plan.run()
        return {"coeffs": s.trace, "evals": s.evals, "layers": s.layers}
    if op == "prove":
        n = case["log"]
        a = s.first.data_ptr()
        proof, _, pos, digest, draws = ctx.wide_fib_prove(a, a + (4 << n), case["cols"], n, s.tw,
                                                          store_coeffs=case["store"])
        # queries may coincide, so a proof's length depends on its inputs
        return {"length": len(proof), "proof": _padded(np.frombuffer(proof, dtype=np.uint8), 1 << 17),
                "positions": _padded(np.array(pos), 8), "digest": np.frombuffer(digest, dtype=np.uint8), "draws": draws}
    if op == "fri":
        roots, last, digest, draws = ctx.fri_commit(s.digest, 0, s.config, s.coords, case["log"], s.tw)
        return {"roots": roots, "last": last, "digest": np.frombuffer(digest, dtype=np.uint8), "draws": draws}
    if op == "interp":
        for c, lg in zip(s.cols, s.logs):
            ctx.bit_reverse_column(c, lg)
        ctx.interpolate_columns(s.cols, s.logs, s.tw)
        return {"coeffs": s.trace}
    if op == "evaluate":
        ctx.evaluate_polynomials(s.cols, s.logs, case["blowup"], s.tw, s.outs)
        return {"evals": s.evals}
    if op == "open":
        values = ctx.eval_at_point(s.cols, s.logs, s.point)
        x, y = s.point
        ctx.compute_fri_quotients(s.outs, s.out_logs, [[(x, y, v)] for v in values.tolist()], s.alpha, s.lifting,
                                  _views(s.quotients, [s.lifting] * 4))
        return {"values": values, "quotients": s.quotients}
    s.server.hold(True)
    ids = []
    for (n, lg, b), t in zip(s.jobs, s.traces):
        ids.append(s.server.submit(n, lg, b, 0, sh.FriConfig(b, 2, 3, 1), cols=_views(t, [lg] * n)))
    s.server.hold(False)
    res = [s.server.wait(i) for i in ids]
    return {"status": np.array([r.status for r in res]),
            "trace_roots": np.array([list(r.trace_root) for r in res], dtype=np.int64),
            "fri_roots": np.array([v for r in res for v in r.fri_roots[: 8 * r.n_fri_roots]], dtype=np.int64),
            "last": np.array([list(r.last_layer_poly[:16]) for r in res], dtype=np.int64),
            "digests": np.array([list(r.final_digest) for r in res])}


# ---- the work a pass cannot do without -----------------------------------------
# Bytes: each input read and each output written once.  Operations: 32-bit
# integer ones; a butterfly is a product, a sum and a difference, a Blake2s
# compression 80 quarter-rounds of 12 (three-input adds counted once).

COMPRESSION = 960
QM31_MUL = 9 * 3


def _fft_ops(lg):
    return 3 * lg * (1 << lg) / 2


def _lde_ops(lg, b):
    return _fft_ops(lg) + (1 << b) * _fft_ops(lg)


def _tree_ops(logs, lifted):
    top = max(logs)
    per = [0] * (top + 1)
    for lg in logs:
        per[top if lifted else lg] += 1
    ops = 0
    for lg in range(top + 1):
        ops += COMPRESSION * (1 << lg) * ((1 if lg < top else 0) + (per[lg] + 15) // 16)
    return ops


def _fri_work(lg, end):
    """Bytes and operations of committed layers of 2^lg, 2^(lg-1), ..."""
    by = ops = 0
    while lg > end:
        by += 16 * (1 << lg) + 64 * (1 << lg)
        ops += 2 * COMPRESSION * (1 << lg) + (1 << (lg - 1)) * (QM31_MUL + 4 * 3)
        lg -= 1
    return by, ops


def work(case):
    op = case["op"]
    if op in ("commit", "batch", "interp", "evaluate", "open"):
        logs = _logs(case)
        b = case.get("blowup", 0)
        words = sum(1 << lg for lg in logs)
        outs = words << b
        top = max(logs) + b
        tree = 4 * sh.tree_words(top)
    if op == "commit":
        by = 4 * outs + tree + (8 * words if case["store"] else 8 << case["lo"])
        ops = sum(_lde_ops(lg, b) for lg in logs) + _tree_ops([lg + b for lg in logs], case["lifted"])
        return {"bytes": by, "flops": ops}
    if op == "batch":
        ops = sum(_lde_ops(lg, b) for lg in logs) + _tree_ops([lg + b for lg in logs], False)
        return {"bytes": 8 * words + 4 * outs + tree, "flops": ops}
    if op == "interp":
        return {"bytes": 8 * words, "flops": sum(_fft_ops(lg) for lg in logs)}
    if op == "evaluate":
        return {"bytes": 4 * words + 4 * outs, "flops": sum((1 << b) * _fft_ops(lg) for lg in logs)}
    if op == "open":
        return {"bytes": 4 * words + 4 * outs + (16 << top), "flops": 3 * 4 * words + 3 * 4 * outs}
    if op == "prove":
        n, c = case["log"], case["cols"]
        fb, fo = _fri_work(n + 1, 1)
        words = (c + 8) << (n + 1)
        ops = c * _lde_ops(n, 1) + 8 * _lde_ops(n, 1) + 2 * COMPRESSION * (2 << n) * ((c + 15) // 16 + 2) / 2
        ops += (c << (n + 1)) * 3 * (1 + 4 + 4) + (c << n) * 12 + fo
        return {"bytes": 4 * words + 4 * 32 * (4 << n) / 2 + 8 * (1 << n) + fb, "flops": ops}
    if op == "fri":
        fb, fo = _fri_work(case["log"], case["last"] + case["blowup"])
        return {"bytes": fb, "flops": fo}
    by = ops = 0
    for n, lg, b in _job_list(case):
        fb, fo = _fri_work(lg + b, b + 2)
        by += 4 * (n << lg) + 4 * (n << (lg + b)) + 4 * sh.tree_words(lg + b) + fb
        ops += n * _lde_ops(lg, b) + _tree_ops([lg + b] * n, True) + fo
    return {"bytes": by, "flops": ops}


def exact(case, seed):
    """Whole numbers only: there is no value in 64 bits to be nearer to."""
    return None
