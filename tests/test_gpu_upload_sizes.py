"""Calls whose column tables lie on both sides of the sizes at which an upload travels
otherwise (256 bytes, 1 KB, 3.5 KB and 7 KB as kernel arguments, more as a copy), one call
after another with no wait in between, against the oracle."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu


def test_tables_one_after_another():
    n, counts = 4, [65, 80, 96, 224, 225, 240, 255, 256, 448, 449, 700]
    evs = [oracle.fill_random(1 << n, 21, c) for c in range(max(counts))]
    with sh.Context(0) as ctx:
        buf = ctx.to_device(np.concatenate(evs))
        cols = [buf.at(c << n) for c in range(max(counts))]
        outs = [ctx.alloc(8 << n) for _ in counts]
        for _ in range(3):
            for C, o in zip(counts, outs):
                ctx.commit_on_layer(n, None, cols[:C], o)
        for C, o in zip(counts, outs):
            assert np.array_equal(o.download(), oracle.merkle_commit(evs[:C])[sh.layer_offset(n):]), C
