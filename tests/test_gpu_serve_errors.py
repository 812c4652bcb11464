"""A group of jobs that fails while its columns are read (one job names a NULL column):
its jobs report the error, and jobs that then run in the same memory are right."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
import stwo_hip as sh  # noqa: E402

pytestmark = pytest.mark.gpu


def test_group_with_a_null_column():
    n, b, C = 14, 1, 24
    fri = sh.FriConfig(b, 1, 3, 1)
    host = np.concatenate([oracle.fill_random(1 << n, 31, c) for c in range(C)])
    with sh.Context(0) as ctx, sh.Server(0, 64 << 20, 17, 2) as srv:
        buf = ctx.to_device(host)
        cols = [buf.at(c << n) for c in range(C)]
        ctx.sync()
        want = srv.wait(srv.submit(C, n, b, 0, fri, cols=cols)).key()
        assert want[0] == 0
        for _ in range(3):
            srv.hold(True)
            bad = [srv.submit(C, n, b, 0, fri, host=host), srv.submit(C, n, b, 5, fri),
                   srv.submit(C, n, b, 0, fri, cols=cols[:-1] + [None])]
            srv.hold(False)
            assert all(srv.wait(i).status == -1 for i in bad)
            good = [srv.submit(C, n, b, 0, fri, host=host), srv.submit(C, n, b, 0, fri, cols=cols)]
            assert all(srv.wait(i).key() == want for i in good)
        buf.free()
