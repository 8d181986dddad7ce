"""Memory that a server keeps of released tenants goes back to the device (GPU): when asked, when an
allocation outside the server needs it, and before another server takes the free memory as its budget."""
import time

import pytest

import graphzeppelin_amd as gz

pytestmark = pytest.mark.gpu

N = 16_384


def _free():
    """The device's free memory once what was given back earlier has arrived."""
    import torch

    last, same = -1, 0
    while same < 3:
        now = torch.cuda.mem_get_info()[0]
        same, last = (same + 1, now) if now == last else (0, now)
        time.sleep(0.03)
    return last


def _keeping_server():
    import torch

    torch.cuda.empty_cache()
    fp = gz.footprint_bytes(N)
    server = gz.Server(16 * fp, 1)
    for t in [server.admit(N, t) for t in range(3)]:
        server.release(t)
    return server, fp


def test_outside_allocation_gets_it():
    server, fp = _keeping_server()
    before = _free()
    print("server keeps, an instance that no memory holds", flush=True)
    with pytest.raises(gz.GZError):
        gz.CCSketchAlg(1 << 26, 1)  # 1.7 TB
    assert _free() - before > 2 * fp
    server.close()


def test_another_servers_budget_counts_it():
    server, fp = _keeping_server()
    before = _free()
    print("server keeps, another server", flush=True)
    other = gz.Server(0, 1)
    assert other.budget_bytes - before > 2 * fp
    other.close()
    server.close()


def test_trim():
    server, fp = _keeping_server()
    before = _free()
    print("server keeps, trim", flush=True)
    assert 0 < server.kept_bytes <= 3 * fp
    assert server.reserved_bytes == 0
    server.trim()
    assert server.kept_bytes == 0
    assert _free() - before > 2 * fp
    t = server.admit(N, 7)
    assert server.reserved_bytes == fp
    server.release(t)
    assert server.reserved_bytes + server.kept_bytes <= server.budget_bytes
    server.close()
