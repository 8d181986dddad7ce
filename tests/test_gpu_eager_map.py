"""Eager DSU over batches large enough to look updates up in the largest component's bits (GPU): at
and below the size, on a new instance and after a query, with vertices outside the component and pairs
out of range, against exact components."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

from test_gpu_eager import _stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [20_001, 262_145])
@pytest.mark.parametrize("count", [(1 << 20) - 1, 1 << 20, (1 << 20) + 77])
def test_lookup_keeps_exact_components(n, count):
    import torch

    print(f"eager lookup n={n} count={count}", flush=True)
    extra = np.array([[n - 1, n - 2], [n - 3, n - 4], [n - 4, n - 5], [n - 5, n - 1]], dtype=np.uint32)
    first = _stream(n, count - 2, count)
    first = np.concatenate([first[:77], extra[:2], first[77:]])  # a small component outside
    alg = gz.CCSketchAlg(n, 7)

    def ingest(p):
        t = torch.from_numpy(p.astype(np.int64).astype(np.int32)).cuda()
        torch.cuda.synchronize()
        alg.ingest_pairs_device(t.data_ptr(), p.shape[0])
        torch.cuda.synchronize()

    def check(so_far):
        cc = alg.connected_components()
        c, lab = oracle.exact_cc(n, so_far)
        assert cc.size() == c and np.array_equal(cc.canonical_labels(), lab)

    ingest(first)
    assert alg.has_cached_query()
    check(first)
    ingest(first[::-1])  # deletes everything
    assert not alg.has_cached_query()
    check(np.concatenate([first, first]))
    ingest(first)  # from nothing again, now with the query's classes
    assert alg.has_cached_query()
    check(first)
    # joins the small components to each other and, in the middle of a large batch, to the largest
    second = np.concatenate([extra[2:], first[: count - 3], np.array([[n - 1, 0]], dtype=np.uint32)])
    ingest(second)
    check(np.concatenate([first, second]))
