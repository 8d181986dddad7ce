"""A vertex whose edges cancel in its deterministic bucket (GPU): four edges (0, x), (0, x'), (0, y),
(0, y') with x ^ x' == y ^ y' and checksums that cancel too sample ZERO although they are there.  The
vertex bridges two pairs, one of them joined to a large component by one edge, so it has to stay in the
query's lists: once their samples have linked it, all of them reach the rest."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu

N, SEED = 1 << 17, 9


def _cancelling_sets(limit):
    """(x, x', y, y') whose edges to vertex 0 cancel in index and 32-bit checksum, not all at one depth
    of column 0."""
    ids = np.arange(1, N, dtype=np.uint64)  # the index of an edge (0, v) is v
    h = np.zeros(N, dtype=np.uint64)
    h[1:] = oracle.xxh3_len8_many(ids, np.full(ids.size, SEED, dtype=np.uint64))
    low = (h & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    out = []
    for p in range(1, 64):
        v = np.arange(2, N, dtype=np.int64)
        v = v[(v < (v ^ p)) & ((v ^ p) < N)]
        both = low[v] ^ low[v ^ p]
        order = np.argsort(both, kind="stable")
        for k in np.flatnonzero(np.diff(both[order].astype(np.int64)) == 0):
            x, y = int(v[order[k]]), int(v[order[k + 1]])
            four = (x, x ^ p, y, y ^ p)
            depths = {int(low[t] & -low[t].astype(np.int64)) for t in four}
            if len(set(four)) == 4 and len(depths) > 1:
                out.append(four)
    return out[:limit]


SETS = 8


@pytest.mark.parametrize("k", range(SETS))
def test_bridge_of_cancelling_edges(k):
    x, x1, y, y1 = _cancelling_sets(SETS)[k]
    print(f"cancelling edges to {x}, {x1}, {y}, {y1}", flush=True)
    rng = np.random.default_rng(k)
    rest = np.setdiff1d(np.arange(1, N), [x, x1, y, y1])
    ring = np.stack([rest, np.roll(rest, 1)], axis=1)
    many = rest[rng.integers(0, rest.size, (8 * N, 2))]
    few = np.array([(0, x), (0, x1), (0, y), (0, y1), (x, x1), (y, y1), (x, rest[100])])
    pairs = np.concatenate([ring, many[many[:, 0] != many[:, 1]], few])
    pairs = np.unique(np.sort(pairs, axis=1), axis=0).astype(np.uint32)
    count, labels = oracle.exact_cc(N, pairs)
    assert count == 1
    for finish in (True, False):
        alg = gz.CCSketchAlg(N, SEED, gz.CCAlgConfiguration(eager_dsu=False))
        alg.set_round_finish(finish)
        alg.ingest_pairs(pairs)
        cc = alg.connected_components()
        assert cc.size() == 1, (cc.size(), alg.last_query_round_sizes())
