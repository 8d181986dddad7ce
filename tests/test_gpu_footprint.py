"""The footprint that admission goes by is what an instance allocates, within what the device's own
account of free memory can tell (GPU): a twentieth."""
import time

import pytest

import graphzeppelin_amd as gz

pytestmark = pytest.mark.gpu


def _free():
    """The device's free memory once what was given back earlier has arrived."""
    import torch

    last, same = -1, 0
    while same < 5:
        now = torch.cuda.mem_get_info()[0]
        same, last = (same + 1, now) if now == last else (0, now)
        time.sleep(0.05)
    return last


@pytest.mark.parametrize("n,kw", [(1000, {}), (4096, dict(gamma_bytes=8)), (16384, dict(flush_threshold=1 << 18)),
                                  (65536, {}), (262144, dict(tile=64))])
def test_footprint_is_what_is_allocated(n, kw):
    import torch

    cfg = gz.CCAlgConfiguration(**kw)
    fp = gz.footprint_bytes(n, cfg)
    count = 12 if n < 100_000 else 2
    print(f"footprint n={n} {kw} {fp}", flush=True)
    torch.cuda.empty_cache()
    warm = [gz.CCSketchAlg(n, 1, cfg) for _ in range(2)]  # what the runtime keeps for streams is there afterwards
    free = _free()
    algs = [gz.CCSketchAlg(n, 1, cfg) for _ in range(count)]
    used = free - _free()
    print(f"used {used / count:.0f} each", flush=True)
    assert abs(used - count * fp) <= count * fp / 20
    for a in algs + warm:
        a.close()
