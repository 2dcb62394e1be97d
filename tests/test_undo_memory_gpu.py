"""The undo history's device memory: moved to the host on request, given back when the history is
cleared, with undo and redo as before over frames on either side, against the oracle."""
import numpy as np
import pytest

from tests.test_edit_gpu import BOX_CARVE, assert_same, make, random_edits

pytestmark = pytest.mark.gpu


def free_bytes():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def wide_pass(p):
    """A carve in the air over many colour subtrees (8 voxels a side), and the bytes of its frame's
    room: a record of 136 bytes for every one its box overlaps inside the scene, and a quarter more."""
    c, r = (p.footprint / 2, 2000.0, p.footprint / 2), 300.0
    boxes = int(np.prod([int((v + r) // 8) - int(max(v - r, 0.0) // 8) + 1 for v in c]))
    return (BOX_CARVE, c, r), boxes * 136 * 5 // 4


def test_history_moves_to_the_host_and_back():
    from tests.test_graph_gpu import canonical
    p, sc, g, dag, od, oc = make("d13")
    wide, room = wide_pass(p)
    lists = [random_edits(p, 1, seed=5), random_edits(p, 30, seed=6), [wide], random_edits(p, 9, seed=7)]
    states = [canonical(dag)]
    for edits in lists:
        dag.edit_batch(edits, fused=True)
        for kind, c, r in edits:
            od.edit(kind, c, r, oc)
        states.append(canonical(dag))
    dag.undo()  # frames to undo and to redo
    held = free_bytes()
    dag.undo_to_host()
    assert free_bytes() - held >= room
    assert dag.undo_depth() == (3, 1)
    dag.undo_to_host()  # nothing left to move
    for k in (2, 1, 0):
        dag.undo()
        assert np.array_equal(canonical(dag), states[k])
    for k in (1, 2, 3, 4):
        dag.redo()
        assert np.array_equal(canonical(dag), states[k])
    assert_same(dag, sc, od, oc, "redone from the host")
    last = random_edits(p, 12, seed=8)  # a frame on the device above frames on the host
    dag.edit_batch(last, fused=True)
    for _ in range(2):
        for _ in range(5):
            dag.undo()
        assert np.array_equal(canonical(dag), states[0])
        for _ in range(5):
            dag.redo()
    for kind, c, r in last:
        od.edit(kind, c, r, oc)
    assert_same(dag, sc, od, oc, "redone from both")


def test_clearing_the_history_gives_its_memory_back():
    p, sc, g, dag, od, oc = make("d13")
    wide, room = wide_pass(p)
    dag.edit_batch([wide])  # grows the scratch too
    before = free_bytes()
    dag.clear_undo()
    assert free_bytes() - before >= room
    cleared = free_bytes()
    for k in range(3):  # small passes live in what stays
        dag.edit_batch(random_edits(p, 4, seed=20 + k), fused=True)
        dag.clear_undo()
    assert cleared - free_bytes() <= 32 << 20
    assert dag.undo_depth() == (0, 0)


def test_an_allocation_without_room_takes_the_histories():
    """A request beyond any card's memory is refused after the history has made room; undo, redo and
    later passes go on."""
    from hashdag_amd._lib import HashDAGError
    from tests.test_graph_gpu import canonical
    p, sc, g, dag, od, oc = make("d13")
    wide, room = wide_pass(p)
    states = [canonical(dag)]
    for edits in (random_edits(p, 10, seed=9), [wide]):
        dag.edit_batch(edits, fused=True)
        for kind, c, r in edits:
            od.edit(kind, c, r, oc)
        states.append(canonical(dag))
    before = free_bytes()
    with pytest.raises(HashDAGError):
        dag.reserve_edit_scratch(16, 16, 1 << 36)  # 512 GiB of staged colours
    assert free_bytes() - before >= room
    for k in (1, 0):
        dag.undo()
        assert np.array_equal(canonical(dag), states[k])
    dag.redo()
    dag.redo()
    more = random_edits(p, 10, seed=10)
    dag.edit_batch(more, fused=True)
    for kind, c, r in more:
        od.edit(kind, c, r, oc)
    assert_same(dag, sc, od, oc, "after the refused request")
