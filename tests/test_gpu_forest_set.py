"""The set of spanning-forest edges at its edges (GPU): tables smaller than one step of its probes, and
tables as full as they get (a tree: every edge is a forest edge).  The cached answer stands until a
forest edge is deleted (pre_insert, src/cc_sketch_alg.cpp:79-104), whichever edge it is."""
import numpy as np
import pytest

import graphzeppelin_amd as gz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("after_query", [False, True])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 9, 64, 1024, 4097])
def test_every_tree_edge_is_in_the_set(n, after_query):
    print(f"forest set n={n} after_query={after_query}", flush=True)
    rng = np.random.default_rng(n)
    perm = rng.permutation(n).astype(np.uint32)
    up = np.array([perm[rng.integers(0, i)] for i in range(1, n)], dtype=np.uint32)
    tree = np.stack([up, perm[1:]], axis=1)
    for k in rng.permutation(n - 1)[:12]:
        alg = gz.CCSketchAlg(n, 3 * n + 1)
        alg.ingest_pairs(tree)
        if after_query:  # the query's forest is the tree; the next batch puts it into the set
            u, v = tree[k]
            alg.pre_insert(int(u), int(v))  # a deletion, as far as the eager DSU knows
            assert not alg.has_cached_query()
            assert alg.connected_components().size() == 1
        assert alg.has_cached_query()
        if n > 2:  # an edge that is not of the tree, inserted and deleted
            known = {(min(a, b), max(a, b)) for a, b in tree.tolist()}
            a, b = next(((a, b) for a in range(n) for b in range(a + 1, n) if (a, b) not in known))
            alg.ingest_pairs(np.array([[a, b], [a, b]], dtype=np.uint32))
            assert alg.has_cached_query()
        alg.ingest_pairs(tree[k:k + 1])
        assert not alg.has_cached_query()
        assert alg.connected_components().size() == 2
