"""The sketch digest at its edges (GPU): fewer vertices than a chunk, chunks that do not divide the
vertex count, bucket counts around a multiple of 64, both checksum widths.  It must be the digest of
the oracle's sketch image."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gb", [4, 8])
@pytest.mark.parametrize("n", [2, 3, 7, 8, 9, 17, 100, 513, 1000, 4099])
def test_digest_of_oracle_image(n, gb):
    print(f"digest n={n} gb={gb}", flush=True)
    rng = np.random.default_rng(n)
    pairs = rng.integers(0, n, (4 * n, 2)).astype(np.uint32)
    pairs = pairs[pairs[:, 0] != pairs[:, 1]]
    seed = 11 * n + gb
    nb = oracle.calc_cc_samples(n, 1.0) * oracle.calc_bkt_per_col(oracle.calc_vector_length(n)) + 1
    ref = oracle.CCAlg(n, seed, gamma_bytes=gb, eager=False)
    ref.ingest_pairs(pairs)
    alg = gz.CCSketchAlg(n, seed, gz.CCAlgConfiguration(eager_dsu=False, gamma_bytes=gb))
    alg.ingest_pairs(pairs)
    assert alg.digest() == gz.digest_of_image(ref.dump(), nb, gb)
