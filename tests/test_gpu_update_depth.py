"""The update kernel's LDS delta (GPU), whose depth follows from the column count: 18 to 28 columns in
one write-back pass, more in several; tiles of a few updates, of nearly and more than a chunk of 64, and
vertices split over tiles; enough edges that buckets past the delta and past the deep flags are
reached.  Every sketch must be the oracle's, bit for bit."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu

N = 1000  # 20 depths


@pytest.mark.parametrize("gb", [4, 8])
@pytest.mark.parametrize("cols", [18, 19, 21, 23, 25, 26, 28, 29, 40])
def test_images_by_column_count(cols, gb):
    factor = (cols - 0.5) / oracle.calc_cc_samples(N, 100.0) * 100.0
    assert oracle.calc_cc_samples(N, factor) == cols
    print(f"update depth cols={cols} gb={gb}", flush=True)
    rng = np.random.default_rng(cols + gb)
    ref = oracle.CCAlg(N, cols, sketches_factor=factor, gamma_bytes=gb, eager=False)
    alg = gz.CCSketchAlg(N, cols, gz.CCAlgConfiguration(sketches_factor=factor, gamma_bytes=gb, eager_dsu=False))
    dense = rng.integers(0, N, (60_000, 2))
    hub = np.stack([np.full(3 * N, 7), rng.integers(0, N, 3 * N)], axis=1)
    for pairs in (rng.integers(0, N, (N, 2)), dense, hub):
        pairs = pairs[pairs[:, 0] != pairs[:, 1]].astype(np.uint32)
        alg.ingest_pairs(pairs)
        ref.ingest_pairs(pairs)
        assert np.array_equal(alg.dump_sketches(0, N), ref.dump())
