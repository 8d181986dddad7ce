"""The segmented reduce's larger shapes at their edges (GPU): rounds of up to 65536 entries take 16 of
them a wave, up to 131072 (or half the vertices) 32, and more than that 64, so lists here end around those
limits and around a wave, a workgroup of 512 and of 1024 entries past them; supernodes lie inside a row,
cross rows, waves and workgroups, or cover several workgroups, and deleted edges come first.  Rounds,
per-round sizes and the partition must be those of a CPU restatement over the edges."""
import numpy as np
import pytest
from scipy.sparse import coo_matrix
from scipy.sparse.csgraph import connected_components

import graphzeppelin_amd as gz
import oracle

pytestmark = pytest.mark.gpu


def _labels(n, a, b):
    return connected_components(coo_matrix((np.ones(a.size, dtype=np.int8), (a, b)), shape=(n, n)), directed=False)[1]


def _partitions(n, edges, D, seed, max_rounds, gb):
    """Labels after rounds 0, 1, ... until one changes nothing: every supernode's bucket is the XOR of its
    cut edges in it (the inner ones cancel), the deterministic bucket's of all of them."""
    idx = (edges.min(axis=1).astype(np.uint64) << np.uint64(32)) | edges.max(axis=1).astype(np.uint64)
    mask = np.uint64(0xFFFFFFFF if gb == 4 else 0xFFFFFFFFFFFFFFFF)

    def hashes(x, s):
        return oracle.xxh3_len8_many(x, np.full(x.size, s, dtype=np.uint64))

    u, v, chk = edges[:, 0].astype(np.int64), edges[:, 1].astype(np.int64), hashes(idx, seed) & mask
    lab, out = np.arange(n), []
    for r in range(max_rounds):
        h = hashes(idx, seed + 5 * r)
        depth = np.full(h.size, D)
        for d in range(D - 1, -1, -1):
            depth[(h & np.uint64((1 << (d + 1)) - 1)) == np.uint64(1 << d)] = d
        k = int(lab.max()) + 1
        alpha, gamma = (np.zeros((k, D + 1), dtype=np.uint64) for _ in range(2))
        cut = lab[u] != lab[v]
        for end in (u, v):
            for where in (depth, np.full(h.size, D)):  # D: no bucket of the column; its place holds the deterministic one
                m = cut & ((where < D) | (where is not depth))
                np.bitwise_xor.at(alpha, (lab[end][m], where[m]), idx[m])
                np.bitwise_xor.at(gamma, (lab[end][m], where[m]), chk[m])
        good = (hashes(alpha.ravel(), seed) & mask).reshape(alpha.shape) == gamma
        zero = (alpha[:, D] == 0) & (gamma[:, D] == 0)
        first = np.where(good[:, D], D, np.argmax(good[:, :D], axis=1))
        found = good.any(axis=1) & ~zero
        picked = alpha[np.arange(k), first][found]
        a, b = (picked >> np.uint64(32)).astype(np.int64), (picked & np.uint64(0xFFFFFFFF)).astype(np.int64)
        assert a.size == 0 or max(a.max(), b.max()) < n
        new = _labels(k, lab[a], lab[b])[lab]
        modified = bool((~found & ~zero).any()) or int(new.max()) != int(lab.max())
        lab = new
        out.append(lab)
        if not modified:
            break
    return out


def _edges(n, shape, rng):
    perm = rng.permutation(n)
    if shape == "path":  # supernodes of every size, doubling round by round
        return np.stack([perm[:-1], perm[1:]], axis=1)
    # trees of 1 to 40 vertices, or of up to 5000, which no majority joins
    cuts = np.cumsum(rng.integers(1, 41 if shape == "small" else 5000, n))
    e = []
    for part in np.split(perm, cuts[cuts < n]):
        up = (rng.random(part.size) * np.arange(part.size)).astype(np.int64)
        e.append(np.stack([part[1:], part[up[1:]]], axis=1))
    return np.concatenate(e)


SIZES = [65_536, 65_537, 65_536 + 511, 65_536 + 513, 98_304 + 31, 131_072, 131_073, 131_072 + 63, 131_072 + 65,
         131_072 + 1023, 131_072 + 1025]


@pytest.mark.parametrize("n,gb", [(n, 4) for n in SIZES] + [(n, 8) for n in SIZES[1::4]])
def test_rounds_at_shape_edges(n, gb):
    seed = 3 * n + gb
    D = oracle.calc_bkt_per_col(oracle.calc_vector_length(n))
    C = oracle.calc_cc_samples(n, 1.0)
    for shape in ("path", "small", "trees"):
        print(f"reduce n={n} gb={gb} {shape}", flush=True)
        rng = np.random.default_rng(seed)
        edges = _edges(n, shape, rng)
        gone = rng.integers(0, n, (n // 2, 2))
        gone = gone[gone[:, 0] != gone[:, 1]]
        parts = _partitions(n, edges, D, seed, C, gb)
        alg = gz.CCSketchAlg(n, seed, gz.CCAlgConfiguration(eager_dsu=False, gamma_bytes=gb))
        for stream in (gone, edges, gone):
            alg.ingest_pairs(stream.astype(np.uint32))
        cc = alg.connected_components()
        assert alg.last_query_rounds == len(parts) - 1
        assert np.array_equal(cc.canonical_labels(), oracle.canonical(parts[-1]))
        for r, (regrouped, giant) in enumerate(alg.last_query_round_sizes(), start=1):
            prev = parts[r - 1]
            assert regrouped == (n if giant is None else n - int(np.count_nonzero(prev == prev[giant]))), r
        alg.close()
