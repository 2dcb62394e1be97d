"""Passes whose upper levels run in one workgroup: editor counts on both sides of each limit (8
editors: filtered a wavefront per slot; 64: a bit each), clustered in one spot and spread out,
with covers at the end and in the middle of the list, against the oracle."""
import numpy as np
import pytest

from tests.test_edit_gpu import BOX_ADD, BOX_CARVE, SPHERE_ADD, SPHERE_CARVE, SPHERE_PAINT, assert_same, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 33, 63, 64, 65])
@pytest.mark.parametrize("name,spread", [("d13", 12.0), ("d13", 200.0), ("d8", 6.0), ("d10w", 90.0)])
def test_clustered_editors_match_oracle(name, spread, n):
    from hashdag_amd import terrain_height
    p, sc, g, dag, od, oc = make(name)
    rng = np.random.default_rng(n * 7 + int(spread))
    F = p.footprint
    x0, z0 = F // 2, F // 3
    edits = []
    for k in range(n):
        x = float(np.clip(round(x0 + rng.uniform(-spread, spread)), 0, F - 1))
        z = float(np.clip(round(z0 + rng.uniform(-spread, spread)), 0, F - 1))
        y = float(terrain_height(p, int(x), int(z)))
        kind = int(rng.choice([SPHERE_ADD, SPHERE_CARVE, BOX_ADD, BOX_CARVE, SPHERE_PAINT]))
        edits.append((kind, (x, y, z), float(round(rng.uniform(1.0, 9.0)))))
    if n > 2:  # whole nodes covered by an editor in the middle, and by the last one
        edits[n // 2] = (BOX_ADD, edits[n // 2][1], 20.0)
        edits[-1] = (BOX_CARVE, edits[-1][1], 11.0)
    st = dag.edit_batch(edits, fused=True)
    total = sum(od.edit(kind, c, r, oc)[1] for kind, c, r in edits)
    assert st.passes == 1 and st.num_voxels == total
    assert_same(dag, sc, od, oc, f"{n} editors")
    dag.undo()  # and again over the nodes the first pass added
    assert dag.edit_batch(edits, fused=True).num_voxels == total
    assert_same(dag, sc, od, oc, f"{n} editors again")
