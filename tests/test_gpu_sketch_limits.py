"""The widest sketches (GPU): the column limit is where it has always been, 424 columns with 4-byte
checksums and 343 with 8-byte ones, for standalone sketches and for a graph's; one column more is
refused, and at the limit both kernels give the oracle's image."""
import math

import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu

LIMIT = {4: 424, 8: 343}


@pytest.mark.parametrize("gb", [4, 8])
def test_standalone_limit(gb):
    print(f"sketch limit gb={gb}", flush=True)
    top = LIMIT[gb]
    for samples, cols in ((top + 1, 1), ((top + 2) // 2, 2), (top + 40, 1)):
        with pytest.raises(gz.GZError):
            gz.Sketch(1 << 40, 1, samples, cols, gb)
    s, r = gz.Sketch(1 << 40, 1, top, 1, gb), oracle.Sketch(1 << 40, 1, top, 1, gb)
    idx = np.random.default_rng(gb).integers(0, 1 << 40, 5000, dtype=np.uint64)
    for part in (idx[:1], idx[1:70], idx):
        s.update_batch(part)
        r.update_batch(part)
        assert s.serialize() == r.serialize()


@pytest.mark.parametrize("gb", [4, 8])
def test_graph_limit(gb):
    n, top = 300, LIMIT[gb]

    def factor(columns):
        f = (columns - 0.5) * (1 - math.log2(1.2)) / math.log2(n)
        assert gz.calc_cc_samples(n, f) == columns
        return f

    print(f"graph limit gb={gb}", flush=True)
    for columns in (top + 1, top + 40):
        with pytest.raises(gz.GZError):
            gz.CCSketchAlg(n, 5, gz.CCAlgConfiguration(gamma_bytes=gb, sketches_factor=factor(columns)))
    pairs = np.random.default_rng(3).integers(0, n, (4000, 2)).astype(np.uint32)
    pairs = pairs[pairs[:, 0] != pairs[:, 1]]
    alg = gz.CCSketchAlg(n, 5, gz.CCAlgConfiguration(gamma_bytes=gb, sketches_factor=factor(top)))
    ref = oracle.CCAlg(n, 5, gamma_bytes=gb, sketches_factor=factor(top))
    alg.ingest_pairs(pairs)
    ref.ingest_pairs(pairs)
    assert np.array_equal(alg.dump_sketches(), ref.dump())
    count, labels = oracle.exact_cc(n, pairs)
    cc = alg.connected_components()
    assert cc.size() == count and np.array_equal(cc.canonical_labels(), labels)
