"""The segmented colour encoder and the edited-voxel count at the sizes where they change path:
colour arrays that end at, just before and just after a segment (4096 colours), arrays of up to and
of more segments than a lane walks on its own (8), a wavefront's tasks of both kinds together, and
editors that leave the scene or fall between voxels. Checked against the oracle, word by word."""
import numpy as np
import pytest

from tests.test_edit_gpu import BOX_ADD, BOX_CARVE, SPHERE_ADD, SPHERE_CARVE, SPHERE_PAINT, assert_same, make

pytestmark = pytest.mark.gpu


# a box of integer centre and radius r holds (2 r)^3 voxels: 4096 at r = 8, 32768 (8 segments) at 16
@pytest.mark.parametrize("r", [7.5, 8.0, 8.5, 16.0, 16.5, 25.0])
@pytest.mark.parametrize("where", ["air", "ground"])
def test_segment_edges_match_oracle(r, where):
    from hashdag_amd import terrain_height
    p, sc, g, dag, od, oc = make("d10w")
    shift = 0.5 if r != int(r) else 0.0  # whole voxels either way
    x, z = 192.0, 192.0  # inside one 128^3 colour subtree
    y = 960.0 if where == "air" else float(terrain_height(p, 192, 192))
    c = (x + shift, y + shift, z + shift)
    edits = [(BOX_ADD, c, r), (SPHERE_PAINT, (x + r, y + r, z + r), r)]  # one colour, then a corner of many
    st = dag.edit_batch(edits, fused=True)
    total = sum(od.edit(kind, cc, rr, oc)[1] for kind, cc, rr in edits)
    assert st.num_voxels == total
    assert_same(dag, sc, od, oc, f"box of radius {r} in the {where}")


@pytest.mark.parametrize("one", [None, BOX_CARVE, BOX_ADD])
def test_one_colour_around_a_segment_matches_oracle(one):
    """4096 colours in a subtree, and one less and one more."""
    p, sc, g, dag, od, oc = make("d10w")
    edits = [(BOX_ADD, (192.0, 960.0, 192.0), 8.0)]
    if one is not None:  # the box's last voxel, or the one beside its face
        edits.append((one, (199.5, 967.5, 199.5) if one == BOX_CARVE else (200.5, 960.5, 192.5), 0.5))
    st = dag.edit_batch(edits, fused=True)
    assert st.num_voxels == sum(od.edit(kind, c, r, oc)[1] for kind, c, r in edits)
    assert st.colors_encoded == 4096 + {None: 0, BOX_CARVE: -1, BOX_ADD: 1}[one]
    assert_same(dag, sc, od, oc, "around a segment")


def test_tasks_of_few_and_many_segments_in_one_wavefront():
    """40 colour subtrees in one workgroup's four wavefronts: more than 8 tasks each, so lanes walk
    arrays of up to 8 segments on their own, beside one of 9 and one of 64 segments."""
    p, sc, g, dag, od, oc = make("d10w")
    dag.set_edit_launch(1 << 30)
    sides = [2, 6, 16, 17, 25, 32] * 6 + [12, 20, 33, 64]  # voxels a side: 1 to 8 segments, 9, 64
    assert sorted({(s ** 3 + 4095) // 4096 for s in sides})[-3:] == [8, 9, 64]
    edits = []
    for k, s in enumerate(sides):  # a subtree each, in the air: 128 voxels a side, 8 along x
        half = s / 2
        at = (128.0 * (k % 8) + 64, 448.0 + 128 * (k // 32), 128.0 * (k // 8 % 4) + 64)
        c = tuple(v + (0.5 if s % 2 else 0.0) for v in at)
        edits.append((BOX_ADD, c, half))
        if k % 3 == 0:  # colours of their own in a corner
            edits.append((SPHERE_PAINT, tuple(v + half for v in c), half))
    st = dag.edit_batch(edits, fused=True)
    assert st.passes == 1
    assert st.num_voxels == sum(od.edit(kind, c, r, oc)[1] for kind, c, r in edits)
    assert_same(dag, sc, od, oc, "few and many segments")


@pytest.mark.parametrize("seed", range(3))
def test_voxel_counts_of_odd_editors(seed):
    p, sc, g, dag, od, oc = make("d8")
    rng = np.random.default_rng(seed)
    edits = []
    for kind in (SPHERE_ADD, SPHERE_CARVE, SPHERE_PAINT, BOX_ADD, BOX_CARVE):
        for r in (0.25, 0.5, 1.0, 1.7, 19.3, 40.0):
            c = rng.uniform(-8.0, 264.0, size=3)  # past the scene's ends too
            if r in (0.5, 40.0):
                c = np.round(c)
            edits.append((kind, tuple(float(np.float32(v)) for v in c), r))
    edits.append((SPHERE_ADD, (300.0, 128.0, 128.0), 20.0))  # touches nothing
    st = dag.edit_batch(edits, fused=True)
    assert st.num_voxels == sum(od.edit(kind, c, r, oc)[1] for kind, c, r in edits)
    assert_same(dag, sc, od, oc, "odd editors")
