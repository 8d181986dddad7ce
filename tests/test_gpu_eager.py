"""Eager DSU over large batches on an MI355X: batches below, at and above the size from which a fresh
instance's batch is ranked and merged in several launches, and batches after a query, against exact
components and the reference's rule (pre_insert, src/cc_sketch_alg.cpp:79-104: the cached answer
stands until an edge of the spanning forest is deleted)."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu


def _stream(n, count, seed):
    """Distinct edges among the first 3n/4 vertices: half of them at 16 hubs, half uniform."""
    rng = np.random.default_rng(seed)
    m = 3 * n // 4
    a = np.where(rng.random(3 * count) < 0.5, rng.integers(0, 16, 3 * count), rng.integers(0, m, 3 * count))
    b = rng.integers(0, m, 3 * count)
    key = (np.minimum(a, b) << 32) | np.maximum(a, b)
    key = key[a != b]
    key = key[np.sort(np.unique(key, return_index=True)[1])][:count]
    assert key.size == count
    return np.stack([key >> 32, key & 0xFFFFFFFF], axis=1).astype(np.uint32)


@pytest.mark.parametrize("feed", ["host", "device"])
@pytest.mark.parametrize("count", [8193, 32767, 32768, 32769, 70_001])
def test_large_batches_keep_exact_components(count, feed):
    import torch

    n = 20_000
    print(f"eager batch count={count} feed={feed}", flush=True)
    pairs = _stream(n, count + 40_000, count)
    first, second = pairs[:count], pairs[count:]
    alg = gz.CCSketchAlg(n, 7)

    def ingest(p):
        if feed == "host":
            alg.ingest_pairs(p)
        else:
            t = torch.from_numpy(p.astype(np.int32)).cuda()
            torch.cuda.synchronize()
            alg.ingest_pairs_device(t.data_ptr(), p.shape[0])
            torch.cuda.synchronize()

    def check(so_far):
        cc = alg.connected_components()
        c, lab = oracle.exact_cc(n, so_far)
        assert cc.size() == c and np.array_equal(cc.canonical_labels(), lab)

    ingest(first)
    assert alg.has_cached_query()  # inserts only: the eager DSU answers
    check(first)
    ingest(first[::2])  # deletes half of the edges, forest edges among them
    assert not alg.has_cached_query()
    left = np.concatenate([first, first[::2]])
    check(left)  # this query ranks the vertices
    ingest(second)
    assert alg.has_cached_query()
    check(np.concatenate([left, second]))
