"""Finished components leave a query's member lists (GPU): graphs of many components that finish in
different rounds, isolated vertices among them, on both sides of the single-workgroup finish's size,
and sketches built from one-sided batches, where nothing is left out.  Rounds, per-round
sizes and partitions must be the CPU restatement's over the oracle's sketch images."""
import numpy as np
import pytest

import graphzeppelin_amd as gz
import oracle

from boruvka_rounds import parse_images, partitions

pytestmark = pytest.mark.gpu


def _check(alg, ref, n, seed):
    D = oracle.calc_bkt_per_col(oracle.calc_vector_length(n))
    C = oracle.calc_cc_samples(n, 1.0)
    alpha, gamma = parse_images(ref.dump(), n, C * D + 1, 4)
    parts = partitions(alpha, gamma, D, seed, C, 4)
    alg.pre_insert(0, 1)  # without the eager DSU this drops the cached answer
    cc = alg.connected_components()
    assert alg.last_query_rounds == len(parts) - 1
    assert np.array_equal(cc.canonical_labels(), oracle.canonical(parts[-1]))
    for r, (regrouped, giant) in enumerate(alg.last_query_round_sizes(), start=1):
        prev = parts[r - 1]
        assert regrouped == (n if giant is None else n - int(np.count_nonzero(prev == prev[giant]))), r


def _components(n, rng):
    """Paths of 1, 2, 4, ... vertices over two thirds of the ids, random edges over the rest."""
    ids = rng.permutation(n)
    cut, size, e = 0, 1, []
    while cut + size < 2 * n // 3:
        part = ids[cut:cut + size]
        e.append(np.stack([part[:-1], part[1:]], axis=1))
        cut += size
        size = size * 2 if size < n // 40 else 1
    rest = ids[cut:]
    e.append(rest[rng.integers(0, rest.size, (rest.size * 2 // 3, 2))])
    e = np.concatenate(e)
    return e[e[:, 0] != e[:, 1]].astype(np.uint32)


@pytest.mark.parametrize("n", [40, 1000, 2048, 2049, 4500])
def test_many_components(n):
    for finish in (True, False):
        print(f"finished components n={n} finish={finish}", flush=True)
        seed = n
        alg = gz.CCSketchAlg(n, seed, gz.CCAlgConfiguration(eager_dsu=False))
        alg.set_round_finish(finish)
        ref = oracle.CCAlg(n, seed, eager=False)
        e = _components(n, np.random.default_rng(n))
        for part in (e[::2], e[1::2], e[: e.shape[0] // 3]):  # the last one deletes
            alg.ingest_pairs(part)
            ref.ingest_pairs(part)
            _check(alg, ref, n, seed)


def test_gutter_batches_keep_every_vertex():
    # batches handed over one end at a time: the library cannot know that the other end's follows, so
    # every component stays in the lists
    n, seed = 1200, 8
    e = _components(n, np.random.default_rng(2))
    alg = gz.CCSketchAlg(n, seed, gz.CCAlgConfiguration(eager_dsu=False))
    ref = oracle.CCAlg(n, seed, eager=False)
    ref.allocate_worker_memory(1)
    alg.ingest_pairs(e[::2])
    ref.ingest_pairs(e[::2])
    for a, b in e[1::2].tolist():
        for src, dst in ((a, b), (b, a)):
            alg.apply_update_batch(0, src, [dst])
            ref.apply_update_batch(0, src, [dst])
    _check(alg, ref, n, seed)
