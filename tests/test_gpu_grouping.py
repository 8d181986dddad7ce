"""Grouping a device-resident batch by vertex (GPU), at the edges of its forms: one workgroup up to
6144 updates, the bucket partition above, one-word records up to 2^21 vertices and two-word ones
above; few and many vertices per bin, hubs that take whole bins, vertices split over several tiles.
Sketch images must equal the oracle's."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu


def _pairs(n, count, rng):
    """A third of the updates at vertex 0, a third among the lowest ids, a third anywhere."""
    a = rng.integers(0, n, count)
    a = np.where(np.arange(count) % 3 == 0, 0, np.where(np.arange(count) % 3 == 1, a % min(n, 16), a))
    b = (a + 1 + rng.integers(0, n - 1, count)) % n
    return np.stack([a, b], axis=1).astype(np.uint32)


def _ingest_device(alg, pairs):
    import torch

    t = torch.from_numpy(pairs.astype(np.int32)).cuda()
    torch.cuda.synchronize()
    alg.ingest_pairs_device(t.data_ptr(), pairs.shape[0])
    alg.prep_query(gz.KSPANNINGFORESTS)  # never cached: applies what is buffered
    torch.cuda.synchronize()


@pytest.mark.parametrize("tile", [0, 8])
@pytest.mark.parametrize("n", [2, 9, 33, 1000, 5001])
def test_grouped_batches_bit_exact(n, tile):
    rng = np.random.default_rng(n + tile)
    alg = gz.CCSketchAlg(n, 11, gz.CCAlgConfiguration(tile=tile))
    ref = oracle.CCAlg(n, 11, eager=False)
    for count in (1, 1023, 6144, 6145, 8193, 70_001, 1):
        print(f"grouping n={n} tile={tile} count={count}", flush=True)
        p = _pairs(n, count, rng)
        _ingest_device(alg, p)
        ref.ingest_pairs(p)
        assert np.array_equal(alg.dump_sketches(), ref.dump())


def test_pairs_out_of_range_are_skipped_and_reported():
    rng = np.random.default_rng(3)
    for count in (6144, 6145, 30_000):
        n = 1000
        alg = gz.CCSketchAlg(n, 11)
        ref = oracle.CCAlg(n, 11, eager=False)
        p = _pairs(n, count, rng)
        bad = p.copy()
        bad[5, 0] = n
        bad[-1, 1] = 0x7FFFFFFF
        with pytest.raises(gz.GZError):
            _ingest_device(alg, bad)
        ref.ingest_pairs(np.delete(p, [5, count - 1], axis=0))
        assert np.array_equal(alg.dump_sketches(), ref.dump())


@pytest.mark.parametrize("count", [6144, 40_000])
def test_two_word_records(count):
    n = (1 << 21) + 3
    print(f"grouping n={n} count={count}", flush=True)
    cfg = gz.CCAlgConfiguration(sketches_factor=0.1, flush_threshold=1 << 17)
    alg = gz.CCSketchAlg(n, 11, cfg)
    p = _pairs(n, count, np.random.default_rng(count))
    _ingest_device(alg, p)
    vl, cols = gz.calc_vector_length(n), gz.calc_cc_samples(n, 0.1)
    ends, deg = np.unique(p, return_counts=True)
    for v in [0, 1, 15, int(ends[-1]), *ends[np.linspace(16, ends.size - 2, 40).astype(int)].tolist()]:
        inc = p[(p[:, 0] == v) | (p[:, 1] == v)].astype(np.uint64)
        idx = (np.minimum(inc[:, 0], inc[:, 1]) << np.uint64(32)) | np.maximum(inc[:, 0], inc[:, 1])
        s = oracle.Sketch(vl, 11, cols, 1, 4)
        s.update_batch(idx)
        assert alg.dump_sketches(v, 1).tobytes() == s.serialize(), v
