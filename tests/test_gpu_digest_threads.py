"""Digests from several threads at once, and beside queries that check the sketches' sum (GPU): each
call gives the value that it gives alone, and the sum's check is not disturbed."""
import threading

import numpy as np
import pytest

import graphzeppelin_amd as gz

pytestmark = pytest.mark.gpu


def _run(jobs):
    errors = []

    def guard(job):
        try:
            job()
        except BaseException as e:  # noqa: BLE001 (handed to the test)
            errors.append(e)

    threads = [threading.Thread(target=guard, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


def _graph(n):
    pairs = np.random.default_rng(n).integers(0, n, (6 * n, 2)).astype(np.uint32)
    return pairs[pairs[:, 0] != pairs[:, 1]]


def test_digests_overlap():
    alg = gz.CCSketchAlg(20_000, 4)
    alg.ingest_pairs(_graph(20_000))
    want = alg.digest()
    print("digest threads", flush=True)

    def job():
        for _ in range(60):
            assert alg.digest() == want

    _run([job] * 4)


def test_digests_beside_the_sum():
    n = 3000
    alg = gz.CCSketchAlg(n, 4, gz.CCAlgConfiguration(eager_dsu=False))
    alg.set_query_graphs(False)  # nothing may wait on an instance's stream while a query's graph is captured on it
    alg.ingest_pairs(_graph(n))
    zero = np.zeros(alg.sketch_bytes(), dtype=np.uint8)
    alg.connected_components()
    want, rounds = alg.digest(), alg.last_query_round_sizes()
    assert any(giant is not None for _, giant in rounds)
    print("digest beside queries", flush=True)
    done = threading.Event()

    def digests():
        while not done.is_set():
            assert alg.digest() == want

    def queries():
        try:
            for _ in range(40):
                alg.apply_raw_buckets_update(0, zero)  # changes nothing, but the sum has to be checked again
                alg.pre_insert(0, 1)  # without the eager DSU this drops the cached answer
                alg.connected_components()
                assert any(giant is not None for _, giant in alg.last_query_round_sizes())
        finally:
            done.set()

    _run([digests, digests, queries])
