"""compute_fri_quotients' samples as the rows handed to the library (CPU): points that
repeat by object and by value, containers of every kind, and a generator that fills the
same lists anew for each column."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stwo-metal_amd"))
import stwo_hip as sh  # noqa: E402


def _rows(samples):
    return [list(x) + list(y) + list(v) for ss in samples for x, y, v in ss]


def _points(kind, n=3):
    rng = np.random.default_rng(4)
    return [tuple(kind([int(w) for w in rng.integers(0, 1 << 32, 4)]) for _ in range(2)) for _ in range(n)]


@pytest.mark.parametrize("kind", [tuple, list, np.uint32, lambda w: np.array(w, dtype=np.uint64)],
                         ids=["tuple", "list", "uint32", "uint64"])
@pytest.mark.parametrize("outer", [list, tuple])
def test_held_samples(kind, outer):
    if kind is np.uint32:
        kind = lambda w: np.array(w, dtype=np.uint32)  # noqa: E731
    a, b, c = _points(kind)
    same = tuple(kind(list(w)) for w in a)  # a's value in other objects
    v = [kind([7 * k, 1, 2 ** 32 - 1, k]) for k in range(8)]
    samples = outer([[(*a, v[0])], [(*a, v[1]), (*b, v[2])], [], [(*b, v[3]), (a[0], b[1], v[4])],
                     [(*same, v[5]), (*a, v[6]), (*c, v[7])]])
    fl, counts = sh._flat_samples(samples)
    assert counts == [1, 2, 0, 2, 3]
    assert fl.tolist() == [[int(w) for w in r] for r in _rows(samples)]


def test_no_samples():
    for samples in ([], [[], []]):
        fl, counts = sh._flat_samples(samples)
        assert counts == [0] * len(samples) and fl.shape == (1, 12) and not fl.any()


class Refilled:
    """Two samples, each in the same two lists."""

    def __init__(self, x, y, first):
        self.x, self.y, self.first = x, y, first

    def __len__(self):
        return 2

    def __iter__(self):
        for k in range(2):
            self.x[:] = [self.first + k] * 4
            self.y[:] = [self.first + k + 100] * 4
            yield self.x, self.y, [k] * 4


def test_one_object_filled_anew():
    x, y = [0] * 4, [0] * 4

    def columns():
        for k in range(3):
            x[:] = [k] * 4
            y[:] = [k + 100] * 4
            yield [(x, y, [k] * 4)]

    fl, counts = sh._flat_samples(columns())
    assert counts == [1, 1, 1] and fl.tolist() == [[k] * 4 + [k + 100] * 4 + [k] * 4 for k in range(3)]
    fl, counts = sh._flat_samples([Refilled(x, y, 10), Refilled(x, y, 20), [(x, y, [9] * 4)]])
    want = [[f + k] * 4 + [f + k + 100] * 4 + [k] * 4 for f in (10, 20) for k in range(2)]
    assert counts == [2, 2, 1] and fl.tolist() == want + [[21] * 4 + [121] * 4 + [9] * 4]
