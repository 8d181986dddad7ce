"""The segmented reduce of a Borůvka round at its edges (GPU): member counts around a row of 16
lanes, a wave's 64 entries, and a workgroup's 1024, 512 and 256 entries; supernodes that lie inside a
row, cross rows, waves and workgroups, or cover them whole; sketches shallower than a row.  Every
round's partition must be the CPU restatement's over the oracle's sketch images, with every round
launched separately and with the single-workgroup finish."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

from boruvka_rounds import parse_images, partitions

pytestmark = pytest.mark.gpu


def _edges(n, shape, rng):
    perm = rng.permutation(n)
    if shape == "path":  # supernodes of every size, doubling round by round
        e = np.stack([perm[:-1], perm[1:]], axis=1)
    elif shape == "star":  # one supernode over everything
        e = np.stack([np.full(n - 1, perm[0]), perm[1:]], axis=1)
    else:  # cliques of 1 to 40 vertices, some of them joined
        cuts = np.cumsum(rng.integers(1, 41, n))
        e = []
        for part in np.split(perm, cuts[cuts < n]):
            a, b = np.triu_indices(part.size, k=1)
            e.append(np.stack([part[a], part[b]], axis=1))
        e.append(rng.integers(0, n, (max(1, n // 60), 2)))
        e = np.concatenate(e)
        e = e[e[:, 0] != e[:, 1]]
    return e.astype(np.uint32)


@pytest.mark.parametrize("gb", [4, 8])
@pytest.mark.parametrize("n", [2, 5, 16, 17, 63, 64, 65, 130, 255, 257, 513, 1023, 1025, 2100])
def test_rounds_at_list_edges(n, gb):
    seed = 3 * n + gb
    D = oracle.calc_bkt_per_col(oracle.calc_vector_length(n))
    C = oracle.calc_cc_samples(n, 1.0)
    for shape in ("path", "star", "cliques"):
        print(f"reduce n={n} gb={gb} {shape}", flush=True)
        pairs = _edges(n, shape, np.random.default_rng(seed))
        ref = oracle.CCAlg(n, seed, gamma_bytes=gb, eager=False)
        ref.ingest_pairs(pairs)
        alpha, gamma = parse_images(ref.dump(), n, C * D + 1, gb)
        parts = partitions(alpha, gamma, D, seed, C, gb)
        for finish in (False, True):
            alg = gz.CCSketchAlg(n, seed, gz.CCAlgConfiguration(eager_dsu=False, gamma_bytes=gb))
            alg.set_round_finish(finish)
            alg.ingest_pairs(pairs)
            for _ in range(2):  # the first query sizes the second one's launched rounds
                alg.pre_insert(0, 1)  # without the eager DSU this drops the cached answer
                cc = alg.connected_components()
                assert alg.last_query_rounds == len(parts) - 1
                assert np.array_equal(cc.canonical_labels(), oracle.canonical(parts[-1]))
                for r, (regrouped, giant) in enumerate(alg.last_query_round_sizes(), start=1):
                    prev = parts[r - 1]
                    out = n if giant is None else n - int(np.count_nonzero(prev == prev[giant]))
                    assert regrouped == out, (r, alg.last_query_round_sizes())
