"""A server's memory while tenants leave and arrive at once (GPU): what its tenants hold and what it keeps
of released ones stay within the budget, whichever call comes first."""
import ctypes
import threading
import time

import numpy as np
import pytest

import graphzeppelin_amd as gz
from graphzeppelin_amd import _lib

pytestmark = pytest.mark.gpu


def _free():
    """The device's free memory once what was given back earlier has arrived."""
    import torch

    last, same = -1, 0
    while same < 3:
        now = torch.cuda.mem_get_info()[0]
        same, last = (same + 1, now) if now == last else (0, now)
        time.sleep(0.03)
    return last


def test_release_beside_admission():
    import torch

    torch.cuda.empty_cache()
    n, count = 16_384, 4
    cfg = gz.CCAlgConfiguration(eager_dsu=False, flush_threshold=1 << 20)
    fp = gz.footprint_bytes(n, cfg)
    pairs = torch.from_numpy(np.random.default_rng(1).integers(0, n, (1 << 20, 2)).astype(np.int32)).cuda()
    free = _free()
    server = gz.Server(count * fp + 1, 1)
    tenants = [server.admit(n, t, cfg) for t in range(count)]
    for k in range(12):
        print(f"server budget pass {k}", flush=True)
        handle = ctypes.c_void_p()
        _lib._check(_lib.lib().gz_server_tenant_alg(server._h, tenants[0], ctypes.byref(handle)))
        for _ in range(64):  # work that the release has to wait for
            _lib._check(_lib.lib().gz_alg_ingest_pairs_device(handle, pairs.data_ptr(), pairs.shape[0]))
        arrived = []

        def admit():
            while not arrived:
                try:
                    arrived.append(server.admit(n, k, cfg))
                except gz.AdmissionError:
                    pass

        other = threading.Thread(target=admit)
        other.start()
        server.release(tenants.pop(0))
        other.join()
        tenants += arrived
        assert server.reserved_bytes <= server.budget_bytes
        assert free - _free() <= server.budget_bytes + fp // 2
    for t in tenants:
        server.release(t)
    server.close()
