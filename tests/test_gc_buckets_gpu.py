"""A collection over buckets of every length its placement meets. Against the oracle: the usual many
short ones, 64 long ones (several rounds of a block) and fewer buckets than a block lays out. Over a
complete octree of random leaves, every word by a walk: a chip full of blocks whose walking wavefront
runs out of LDS room (65536 buckets of 32 leaves, 2048 a block), and rounds that end within a list."""
from dataclasses import replace

import numpy as np
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


def test_gc_of_a_million_leaves_keeps_every_word():
    from hashdag_amd import Geometry, HashDAG
    levels, L = 9, 7
    rng = np.random.default_rng(11)
    leaves = rng.integers(1, 2 ** 63, size=8 ** L, dtype=np.int64).view(np.uint32).reshape(-1, 2)
    first = [9 * (8 ** l - 1) // 7 for l in range(L + 1)]  # word of a level's first node, breadth first
    words = np.empty(first[L] + 2 * 8 ** L, np.uint32)
    for l in range(L):
        node = np.full((8 ** l, 9), 0xFF, np.uint32)
        node[:, 1:] = (first[l + 1] + (9 if l + 1 < L else 2) * np.arange(8 ** (l + 1))).reshape(-1, 8)
        words[first[l]:first[l + 1]] = node.ravel()
    words[first[L]:] = leaves.ravel()
    g = Geometry(levels=levels, num_top_levels=6, bucket_bits_top=10, bucket_bits_low=16, bucket_size_top=1024,
                 bucket_size_low=1024, color_tree_levels=2)
    with HashDAG(g, pool_pages=1 << 18) as dag:
        dag.load_basic_dag(words)
        for _ in range(2):
            assert dag.remove_stale_nodes()["live_nodes"] == (8 ** (L + 1) - 1) // 7
            img = dag.download()

            def at(va):
                return img.pool[img.page_table[va // g.page_size].astype(np.int64) * g.page_size + va % g.page_size]

            va = np.array([img.root], np.int64)
            for l in range(L):
                assert (at(va) == 0xFF).all(), f"headers of level {l}"
                va = at(va[:, None] + 1 + np.arange(8)).astype(np.int64).ravel()
            assert np.unique(va).size == va.size
            assert np.array_equal(at(va[:, None] + np.arange(2)), leaves)
