"""Sketch::update over a batch (GPU) at the edges of its kernel: less than a wave, one workgroup, the
whole grid and more; sketches shallower than the LDS delta, and with more columns than the deep delta
takes.  Host and device-resident indices must give the oracle's image."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gb", [4, 8])
@pytest.mark.parametrize("vl,samples,cols", [(1, 18, 1), (300, 18, 1), (1 << 20, 19, 1), (1 << 35, 25, 1), (1 << 60, 28, 2),
                                             (1 << 35, 160, 1), (1 << 35, 23, 7)])
def test_batches_bit_exact(vl, samples, cols, gb):
    import torch

    a = gz.Sketch(vl, 9, samples, cols, gb)
    b = gz.Sketch(vl, 9, samples, cols, gb)
    r = oracle.Sketch(vl, 9, samples, cols, gb)
    rng = np.random.default_rng(samples + gb)
    for count in (1, 63, 64, 65, 1023, 1024, 1025, 20_001):
        print(f"sketch update vl={vl} {samples}x{cols} gb={gb} count={count}", flush=True)
        idx = rng.integers(0, vl, count, dtype=np.uint64)
        dev = torch.from_numpy(idx.view(np.int64)).cuda()
        torch.cuda.synchronize()
        a.update_batch(idx)
        b.update_batch_device_noalloc(dev.data_ptr(), count)
        r.update_batch(idx)
        assert a.serialize() == r.serialize() and b.serialize() == r.serialize(), count


def test_more_than_the_grid_bit_exact():
    vl, count = 1 << 35, 512 * 1024 + 77
    s, r = gz.Sketch(vl, 4, 25), oracle.Sketch(vl, 4, 25)
    idx = np.random.default_rng(1).integers(0, vl, count, dtype=np.uint64)
    s.update_batch(idx)
    r.update_batch(idx)
    assert s.serialize() == r.serialize()
