"""Batches of one standalone sketch that are smaller than a workgroup (GPU): counts around the powers of two
at which an index gets fewer lanes, with fewer columns than lanes, as many, and many more.  The image must
be the oracle's after every batch, and the sample with it."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gb", [4, 8])
@pytest.mark.parametrize("columns", [1, 2, 3, 18, 31, 32, 33, 64, 65, 160, 161, 343])
def test_small_batches_bit_exact(columns, gb):
    vl = 1 << 40
    s, r = gz.Sketch(vl, 5, columns, 1, gb), oracle.Sketch(vl, 5, columns, 1, gb)
    rng = np.random.default_rng(columns)
    print(f"small batches columns={columns} gb={gb}", flush=True)
    for count in (1, 2, 15, 16, 17, 31, 32, 33, 127, 129, 256, 257, 511, 512, 513, 1023, 1024, 1025):
        idx = rng.integers(0, vl, count, dtype=np.uint64)
        s.update_batch(idx)
        r.update_batch(idx)
        assert s.serialize() == r.serialize(), count
    for k in range(min(columns, 3)):
        assert s.sample() == r.sample(), k
