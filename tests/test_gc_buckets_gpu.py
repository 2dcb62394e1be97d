"""A collection over buckets of every length its placement meets: the usual many short ones, 64
long ones (more nodes than a block lists in LDS) and fewer buckets than a block lays out, against
the oracle."""
from dataclasses import replace

import pytest

from tests.test_edit_gpu import POOL_PAGES, assert_same, random_edits, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top,low", [(10, 16), (6, 6), (4, 8)])
def test_gc_over_few_long_buckets_matches_oracle(top, low):
    from hashdag_amd import HashDAG
    from oracle import OracleColors, OracleDAG
    p, sc, g = scene("d13")
    g = replace(g, bucket_bits_top=top, bucket_size_top=g.bucket_size_top << max(0, g.bucket_bits_top - top),
                bucket_bits_low=low, bucket_size_low=g.bucket_size_low << max(0, g.bucket_bits_low - low))
    dag = HashDAG(g, pool_pages=POOL_PAGES)
    dag.load_scene(sc)
    od, oc = OracleDAG.from_basic(g, sc.dag, POOL_PAGES), OracleColors.from_scene(sc)
    for kind, center, r in random_edits(p, 5, seed=41):
        dag.edit(kind, center, r)
        od.edit(kind, center, r, oc)
    live = int(OracleDAG.from_image(dag.download(), dag.pool_pages).reachable(g.leaf_level).sum())
    st = dag.remove_stale_nodes()
    od.gc(g.leaf_level)
    assert st["live_nodes"] == live and st["words_after"] < st["words_before"]
    assert_same(dag, sc, od, oc, "after GC")
