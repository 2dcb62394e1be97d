"""A pass whose levels are large enough for the launches that take many slots at a time: expands in
rounds of 1024 slots, colour copies a wavefront per item, runs of one colour in a leaf. Covers of
one colour under later editors of the same pass leave slots whose old colour is one."""
import numpy as np
import pytest

from tests.test_edit_gpu import BOX_ADD, BOX_CARVE, SPHERE_ADD, SPHERE_CARVE, SPHERE_PAINT, assert_same, make

pytestmark = pytest.mark.gpu


def boxed(edits, side, world):
    """nodes of a level that the editors' boxes overlap, each editor's counted: what launches go by"""
    return sum(int(np.prod([int(min(v + r, world) // side) - int(max(v - r, 0) // side) + 1 for v in c]))
               for _, c, r in edits)


@pytest.mark.parametrize("reserved", [False, True])
@pytest.mark.parametrize("last", [SPHERE_CARVE, SPHERE_ADD, SPHERE_PAINT])
def test_wide_overlapping_editors_match_oracle(last, reserved):
    from hashdag_amd import terrain_height
    p, sc, g, dag, od, oc = make("d13")
    F = p.footprint
    x, z = F // 2, F // 3
    y = float(terrain_height(p, x, z))
    edits = []
    for k in range(24):  # boxes of 150 a side bound the pass; spread so little that they overlap
        c = (float(x + 5 * (k % 5)), y + 3.0 * (k % 3), float(z + 4 * (k % 7)))
        edits.append(((SPHERE_ADD, BOX_CARVE, SPHERE_CARVE, BOX_ADD)[k % 4], c, 70.0 + k % 6))
    edits.append((BOX_ADD, (float(x), y, float(z)), 75.0))
    edits.append((last, (float(x + 3), y + 5.0, float(z + 1)), 33.0))
    # the leaves' parents expand in rounds of 1024 slots from 2^17 items by the boxes, where the
    # scratch holds as many (its first size does not)
    assert boxed(edits, 8, 1 << g.levels) >= 1 << 17
    if reserved:
        dag.reserve_edit_scratch(1 << 18, 1 << 20, 1 << 22)
    st = dag.edit_batch(edits, fused=True)
    total = sum(od.edit(kind, c, r, oc)[1] for kind, c, r in edits)
    assert st.passes == 1 and st.num_voxels == total
    assert_same(dag, sc, od, oc, "large levels")
