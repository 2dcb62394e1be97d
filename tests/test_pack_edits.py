"""pack_edits against the field-by-field form: the same bytes for every accepted list, the same
refusals for the others."""
import ctypes as C

import numpy as np
import pytest

from hashdag_amd._lib import hd_edit
from hashdag_amd.dag import fill_edit, pack_edits


def plain(edits):
    arr = (hd_edit * max(len(edits), 1))()
    for i, ed in enumerate(edits):
        fill_edit(arr[i], ed)
    return bytes(arr)


def lists():
    rng = np.random.default_rng(3)
    base = [(int(rng.integers(0, 5)), tuple(float(v) for v in rng.uniform(-10, 1e5, 3)), float(rng.uniform(0.1, 300)))
            for _ in range(40)]
    yield "floats", base
    yield "short", base[:15]
    yield "empty", []
    yield "ints and numpy scalars", [(np.int32(k), np.array(c, np.float32), np.float32(r)) for k, c, r in base]
    yield "integer centres", [(k, [int(v) for v in c], int(r) + 1) for k, c, r in base]
    yield "beyond float32", base[:20] + [(1, (1e300, -1e300, 0.1), 1e39)]
    yield "nan and kinds out of range", base[:20] + [(-1, (float("nan"), 1.0, 2.0), float("nan")), (2 ** 31, (0, 0, 0), 1)]
    yield "copies among them", base[:20] + [(5, (1, 2, 3), 4.0, (1, 2, 3), (7, 8, 9), np.eye(3) * 2, 0.5)]


@pytest.mark.parametrize("name,edits", list(lists()), ids=[n for n, _ in lists()])
def test_same_bytes(name, edits):
    assert bytes(pack_edits(edits)) == plain(edits)
    assert isinstance(pack_edits(edits), C.Array)


@pytest.mark.parametrize("bad", [(0, (1.0, 2.0), 3.0), (0, (1.0,), 3.0), (0, (1.0, 2.0, 3.0, 4.0), 1.0), (0, None, 1.0),
                                 (0, (1.0, 2.0, "x"), 1.0), ("k", (1.0, 2.0, 3.0), 1.0), (0, (1.0, 2.0, 3.0), None),
                                 (0, (1.0, None, 2.0), 3.0), (0, (1.0, np.datetime64("2020"), 2.0), 3.0)])
def test_same_refusals(bad):
    for edits in ([(0, (1.0, 2.0, 3.0), 4.0)] * 30 + [bad], [bad] * 20):
        with pytest.raises(Exception) as want:
            plain(edits)
        with pytest.raises(want.type):
            pack_edits(edits)


def test_numpy_error_state_of_the_caller():
    """Values that leave float32's range pack alike whatever numpy is told to do about it."""
    edits = [(0, (1e-50, 1e300, 2.0), 1e-60)] * 20
    with np.errstate(all="raise"):
        assert bytes(pack_edits(edits)) == plain(edits)


def test_centres_that_are_read_once():
    """A centre that is an iterator is read by one of the forms only."""
    def edits(bad=False):
        return [(0, iter((1.0, 2.0, 3.0)), 4.0) for _ in range(19)] + [(0, (1.0, None if bad else 0.0, 2.0), 3.0)]
    assert bytes(pack_edits(edits())) == plain(edits())
    with pytest.raises(TypeError):
        pack_edits(edits(bad=True))
