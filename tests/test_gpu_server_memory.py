"""Memory of released tenants (GPU): instances on recycled blocks give the oracle's sketches and exact
answers, also when several threads admit and release at once; nothing is held beyond the budget's
unreserved part, and a destroyed server gives everything back."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle
from graphzeppelin_amd import gen

pytestmark = pytest.mark.gpu


def _tenants(ns, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in ns:
        p = rng.integers(0, n, (6 * n, 2)).astype(np.uint32)
        out.append((n, p[p[:, 0] != p[:, 1]]))
    return out


@pytest.mark.parametrize("workers", [1, 4])
def test_recycled_blocks(workers):
    import torch

    server = gz.Server(4 << 30, workers)
    ns = [1000, 1000, 3000, 700, 2049, 1000]
    for seed in range(4):
        print(f"server memory workers={workers} pass={seed}", flush=True)
        ten = _tenants(ns, seed)
        dev = [torch.from_numpy(p.astype(np.int32)).cuda() for _, p in ten]
        torch.cuda.synchronize()
        trace = gen.multi_tenant_trace(ten, seed, None)
        seeds = [10 * seed + t for t in range(len(ns))]
        lat, ans, dig, st, par = server.run_trace(trace, [d.data_ptr() for d in dev], ns, seeds, want_parents=True)
        assert server.reserved_bytes == 0
        for t, (n, p) in enumerate(ten):
            ref = oracle.CCAlg(n, seeds[t], eager=False)
            ref.ingest_pairs(p)
            nb = gz.calc_cc_samples(n) * gz.calc_bkt_per_col(gz.calc_vector_length(n)) + 1
            assert int(dig[t]) == gz.digest_of_image(ref.dump(), nb)
            c, lab = oracle.exact_cc(n, p)
            assert np.array_equal(gz.ConnectedComponents(par[t], c).canonical_labels(), lab)
    server.close()


def test_kept_memory_is_bounded_and_given_back():
    import torch

    torch.cuda.empty_cache()
    n = 50_000
    fp = gz.footprint_bytes(n)
    free0 = torch.cuda.mem_get_info()[0]
    server = gz.Server(8 * fp, 1)
    for _ in range(3):
        ids = [server.admit(n, 1) for _ in range(8)]
        for t in ids:
            server.release(t)
    # at most a quarter of the budget stays with the server
    assert free0 - torch.cuda.mem_get_info()[0] < 2 * fp + (256 << 20)
    ids = [server.admit(n, 1) for _ in range(7)] + [server.admit(n // 2, 1)]
    with pytest.raises(gz.AdmissionError):
        server.admit(n, 1)
    for t in ids:
        server.release(t)
    server.close()
    assert free0 - torch.cuda.mem_get_info()[0] < 256 << 20
