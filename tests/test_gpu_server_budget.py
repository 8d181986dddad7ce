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


def test_admissions_and_releases_at_once():
    sizes = [1000, 4096]
    budget = 6 * gz.footprint_bytes(sizes[1])
    server = gz.Server(budget, 1)
    for phase in range(15):
        print(f"server churn phase {phase}", flush=True)
        errors = []

        def churn(seed):
            rng = np.random.default_rng(seed)
            mine = []
            try:
                for _ in range(40):
                    if mine and rng.random() < 0.5:
                        server.release(mine.pop(int(rng.integers(len(mine)))))
                        continue
                    try:
                        mine.append(server.admit(sizes[int(rng.random() < 0.5)], 1))
                    except gz.AdmissionError:
                        if mine:
                            server.release(mine.pop())
                for t in mine:
                    left.append(t)
            except BaseException as e:  # noqa: BLE001 (handed to the test)
                errors.append(e)

        left = []
        threads = [threading.Thread(target=churn, args=(4 * phase + t,)) for t in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        assert server.reserved_bytes + server.kept_bytes <= budget
        for t in left:
            server.release(t)
        assert server.reserved_bytes == 0 and server.kept_bytes <= budget // 4
    server.close()


def test_one_takes_what_is_kept_while_another_allocates():
    # 30 small tenants and ten kept blocks of their size fill the budget but for 20 MB; a larger tenant, which
    # needs some of the kept memory given back, and a small one, which takes a kept block, arrive at once
    small, large = 1000, 2000
    fp = gz.footprint_bytes(small)
    budget = 40 * fp
    assert gz.footprint_bytes(large) > fp
    server = gz.Server(budget, 1)
    for _ in range(30):
        server.admit(small, 1)
    for k in range(40):
        print(f"server arrivals pass {k}", flush=True)
        server.trim()
        for t in [server.admit(small, 1) for _ in range(10)]:
            server.release(t)
        assert server.kept_bytes > 9 * (fp - (4 << 20))
        arrived, gate = [], threading.Barrier(2)

        def admit(n):
            gate.wait()
            arrived.append(server.admit(n, 1))

        threads = [threading.Thread(target=admit, args=(n,)) for n in (large, small)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(arrived) == 2
        assert server.reserved_bytes + server.kept_bytes <= budget
        for t in arrived:
            server.release(t)
    server.close()
