"""Grouping flushes so large that records move through LDS (GPU): just below and above the size, bins
of few and of more than 1024 vertices, one-word and two-word records, hubs and pairs out of range.
Sketches must equal the oracle's."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

from test_gpu_grouping import _ingest_device, _pairs

pytestmark = pytest.mark.gpu

LARGE = 1 << 22  # updates; twice as many entries


@pytest.mark.parametrize("n", [3, 1000, 5001])
def test_large_flush_bit_exact(n):
    rng = np.random.default_rng(n)
    alg = gz.CCSketchAlg(n, 11, gz.CCAlgConfiguration(flush_threshold=LARGE + 5000))
    ref = oracle.CCAlg(n, 11, eager=False)
    for count in (LARGE - 1, LARGE, LARGE + 4321):
        print(f"large grouping n={n} count={count}", flush=True)
        p = _pairs(n, count, rng)
        _ingest_device(alg, p)
        ref.ingest_pairs(p)
        assert np.array_equal(alg.dump_sketches(), ref.dump())


def test_large_flush_skips_pairs_out_of_range():
    n = 1000
    p = _pairs(n, LARGE + 11, np.random.default_rng(1))
    bad = p.copy()
    at = [0, 4095, 4096, LARGE + 10]
    bad[at, [0, 1, 0, 1]] = [n, 0xFFFFFFF, n + 7, n]
    alg = gz.CCSketchAlg(n, 11, gz.CCAlgConfiguration(flush_threshold=LARGE + 5000))
    with pytest.raises(gz.GZError):
        _ingest_device(alg, bad)
    ref = oracle.CCAlg(n, 11, eager=False)
    ref.ingest_pairs(np.delete(p, at, axis=0))
    assert np.array_equal(alg.dump_sketches(), ref.dump())


@pytest.mark.parametrize("n", [(1 << 20) + 5, (1 << 21) + 3])  # bins of 2048 vertices; two-word records
def test_large_flush_many_vertices(n):
    print(f"large grouping n={n}", flush=True)
    alg = gz.CCSketchAlg(n, 11, gz.CCAlgConfiguration(sketches_factor=0.1, flush_threshold=LARGE + 5000))
    p = _pairs(n, LARGE + 9, np.random.default_rng(n))
    _ingest_device(alg, p)
    vl, cols = gz.calc_vector_length(n), gz.calc_cc_samples(n, 0.1)
    ends = np.unique(p)
    for v in [0, 1, 15, *ends[np.linspace(16, ends.size - 1, 12).astype(int)].tolist()]:
        inc = p[(p[:, 0] == v) | (p[:, 1] == v)].astype(np.uint64)
        idx = (np.minimum(inc[:, 0], inc[:, 1]) << np.uint64(32)) | np.maximum(inc[:, 0], inc[:, 1])
        s = oracle.Sketch(vl, 11, cols, 1, 4)
        s.update_batch(idx)
        assert alg.dump_sketches(v, 1).tobytes() == s.serialize(), v
