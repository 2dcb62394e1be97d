"""Passes that touch more nodes than their editors' boxes overlap. A sphere whose radius is one step
past the distance to a node's upper edge touches that node, while centre - radius rounds onto the
edge, so the box (what a pass's launch forms and its undo frame's room are chosen by) ends there.
Undo frames larger than their room, and levels around the root that outgrow the workgroup that runs
them, against the oracle."""
import numpy as np
import pytest

from tests.test_edit_gpu import SPHERE_ADD, SPHERE_CARVE, SPHERE_PAINT, assert_same, make

pytestmark = pytest.mark.gpu

R = np.nextafter(np.float32(1.0), np.float32(2.0))


def boxed(c, side):
    """nodes of a level that the editor's box overlaps, as the library counts them"""
    lo = [np.float32(v) - R for v in c]
    hi = [np.float32(v) + R for v in c]
    return int(np.prod([int(h // side) - int(l // side) + 1 for l, h in zip(lo, hi)]))


def touched(c, side):
    """nodes of a level that the sphere touches (FP32, in the library's order)"""
    n = 0
    base = [int(v // side) for v in c]
    for d in np.ndindex(5, 5, 5):
        dist = R * R
        for a in range(3):
            v0 = np.float32((base[a] + d[a] - 2) * side)
            v1 = np.float32(v0 + side)
            ca = np.float32(c[a])
            if ca < v0:
                dist = np.float32(dist - (ca - v0) * (ca - v0))
            elif ca > v1:
                dist = np.float32(dist - (ca - v1) * (ca - v1))
        n += bool(dist > 0)
    return n


def places(n):
    return [np.array((64 * (i % 4), 64 * (i // 4 % 4), 64 * (i // 16)), np.float64) + 64 for i in range(n)]


# centre past a place's lower edges, editors, the levels' limit by boxes, what the level grows to
ONE = (np.array((1.0, 35.0, 37.0)), 1, 1, 2)          # the undo frame's room: one colour leaf
NODES = (np.array((1.0, 35.0, 37.0)), 30, 32, 60)     # build and nodes in one workgroup: 32 items
EXPAND = (np.array((1.0, 1.0, 0.0)), 64, 128, 384)    # expand in one workgroup: 128 items, 256 in LDS


@pytest.mark.parametrize("name", ["d13", "d10"])
@pytest.mark.parametrize("shape", [ONE, NODES, EXPAND], ids=["undo frame", "nodes", "expand"])
def test_more_nodes_than_the_boxes_match_oracle(shape, name):
    from tests.test_graph_gpu import canonical
    shift, n, limit, most = shape
    centres = [tuple(float(v) for v in at + shift) for at in places(n)]
    for side in (8, 16, 32):  # the parents of leaves, and nodes above (colour subtrees among them)
        assert sum(boxed(c, side) for c in centres) <= limit
        assert sum(touched(c, side) for c in centres) == most
    p, sc, g, dag, od, oc = make(name)
    before = canonical(dag)
    kinds = (SPHERE_ADD, SPHERE_PAINT, SPHERE_ADD, SPHERE_CARVE) if n > 1 else (SPHERE_ADD,)
    edits = [(kinds[i % len(kinds)], c, float(R)) for i, c in enumerate(centres)]
    st = dag.edit_batch(edits, fused=True)
    ovox = [od.edit(kind, c, r, oc) for kind, c, r in edits]
    assert st.passes == 1 and st.num_voxels == sum(v[1] for v in ovox)
    assert_same(dag, sc, od, oc, "first pass")
    after = canonical(dag)
    dag.undo()
    assert np.array_equal(canonical(dag), before)
    dag.redo()
    assert np.array_equal(canonical(dag), after)
    assert_same(dag, sc, od, oc, "redone")
    dag.undo()  # and again, over nodes and colour leaves that are there
    assert dag.edit_batch(edits, fused=True).num_voxels == st.num_voxels
    assert_same(dag, sc, od, oc, "second pass")
