"""Workloads that the framework's speed is measured on.

Every case is one thing a program does with the library, through its Python entry points: keep a
standalone sketch, keep one graph stream's connected components (fed from device or host memory,
through the driver's plugin interface, or as a served request trace), or serve several streams at
once.  Sizes follow the repository's own configurations (n = 1024, the planted blocks at 2^15, R-MAT
at 2^17, Chung-Lu at 2^18, tenants up to 2^20), with odd sizes beside the powers of two.

Updates toggle edges, so a pass applies a batch of churn to a graph that is already there: half of
the batch deletes present edges and half inserts absent ones, and the next pass on the same state
undoes it, so every pass meets a graph of the same size and shape.  Nothing computed here is a
floating-point number: sketches are XORs of 64-bit indices and 32- or 64-bit checksums, and answers
are counts and truth values.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import graphzeppelin_amd as gz
from graphzeppelin_amd import gen

DEV = "cuda"


def listed():
    return [
        # A short vector sketched on its own: a handful of indices, a sample and the byte image, all latency.
        dict(name="sketch_few", kind="sketch", n=4096, count=48, feed="host", gamma=4),
        # One sketch over a long device-resident vector, through the entry point that allocates nothing.
        dict(name="sketch_bulk", kind="sketch", n=1 << 18, count=4_194_301, feed="device", gamma=4),
        # The smallest graphs (unit tests, one small community): a thousand host updates, all labels.
        dict(name="tiny_graph", kind="graph", model="uniform", n=1000, base=1_500, updates=1_000, feed="host", gamma=4,
             watch=0, ask="labels"),
        # The driver's plugin interface: one gutter per vertex handed to apply_update_batch, then a
        # query and a checkpoint image of every sketch.
        dict(name="plugin_gutters", kind="plugin", n=1024, per_vertex=100, gamma=4),
        # Clusters on a mid-size graph (the planted-blocks configuration): components after half a million updates.
        dict(name="blocks_32k", kind="graph", model="blocks", n=32_749, base=1_000_000, updates=524_288, feed="device",
             gamma=4, watch=4096, ask="cc"),
        # An insert-mostly stream between queries: no forest edge is deleted, so the eager DSU answers.
        dict(name="cached_points", kind="cached", model="chung_lu", n=1 << 18, base=8_000_000, updates=65_536, watch=1024,
             gamma=4),
        # A query soon after the last one: a small batch, then a list of watched pairs that needs Boruvka.
        dict(name="point_after_5k", kind="graph", model="chung_lu", n=1 << 18, base=8_000_000, updates=5_000,
             feed="device", gamma=4, watch=1024, ask="points"),
        # The serving loop: batches of 1k to 1M updates with about one request per 400k updates.
        dict(name="serve_256k", kind="serve", model="chung_lu", n=1 << 18, base=12_000_000, updates=24_000_000,
             per_request=400_000, gamma=4),
        # Bulk loading between rare queries.
        dict(name="bulk_256k", kind="graph", model="chung_lu", n=1 << 18, base=16_000_000, updates=24_000_000,
             feed="device", gamma=4, watch=65_536, ask="cc"),
        # 64-bit checksums, fed from pageable host memory (the R-MAT configuration).
        dict(name="host_rmat_128k_g8", kind="graph", model="rmat", n=1 << 17, base=3_000_000, updates=3_000_000,
             feed="host", gamma=8, watch=4096, ask="cc"),
        # The largest graphs: a million vertices, an odd count, 17 GB of sketches.
        dict(name="rmat_1m", kind="graph", model="rmat", n=1_000_003, base=12_000_000, updates=16_000_000,
             feed="device", gamma=4, watch=65_536, ask="cc"),
        # Several streams of very different sizes served as one mix, admitted and released on the way.
        dict(name="tenants", kind="tenants", tenants=5, log2_lo=12.0, log2_hi=17.0, per_nlogn=2.0, gamma=4),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sketch", "graph", "graph", "graph", "graph", "plugin", "cached", "serve", "tenants"])
    gamma = rng.choice([4, 4, 4, 8])
    if kind == "sketch":
        feed = rng.choice(["host", "device"])
        return dict(kind=kind, n=_logint(rng, 1000, 1 << 20), count=_logint(rng, 1, 4_194_301 if feed == "device" else 300_000),
                    feed=feed, gamma=gamma)
    if kind == "plugin":
        return dict(kind=kind, n=_logint(rng, 200, 2000), per_vertex=rng.randint(3, 150), gamma=gamma)
    if kind == "tenants":
        lo = rng.uniform(10.0, 13.0)
        return dict(kind=kind, tenants=rng.randint(2, 5), log2_lo=lo, log2_hi=rng.uniform(lo + 1.0, 17.0),
                    per_nlogn=rng.uniform(0.5, 2.0), gamma=gamma)
    n = _logint(rng, 1 << 15, 1 << 18)
    if kind == "cached":
        return dict(kind=kind, model="chung_lu", n=n, base=n * rng.randint(16, 30), updates=_logint(rng, 100, 300_000),
                    watch=_logint(rng, 100, 4096), gamma=gamma)
    if kind == "serve":
        base = n * rng.randint(16, 48)
        return dict(kind=kind, model="chung_lu", n=n, base=base, updates=_logint(rng, 1_000_000, 2 * base),
                    per_request=_logint(rng, 200_000, 1_600_000), gamma=gamma)
    model = rng.choice(["uniform", "blocks", "rmat", "chung_lu"])
    n = _logint(rng, 1 << 12, 1 << 19)
    if n >= 1 << 18:
        gamma = 4
    base = max(4 * n, min(16_000_000, n * rng.randint(4, 24)))
    feed = rng.choice(["device", "device", "host"])
    updates = _logint(rng, 100, min(2 * base, 16_000_000 if feed == "device" else 3_000_000))
    return dict(kind=kind, model=model, n=n, base=base, updates=updates, feed=feed, gamma=gamma,
                watch=_logint(rng, 100, 65_536), ask=rng.choice(["cc", "points"]))


# ---- inputs ------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


@functools.lru_cache(maxsize=8)
def _chung_lu_cdf(n):
    """Power-law expected degrees (exponent 2.1, mean 64), summed and normalised."""
    cdf = np.cumsum(gen.chung_lu_weights(n, 2.1, 64.0))
    return cdf / cdf[-1]


def _candidates(case, count, g):
    """Edge keys (min << 32 | max) drawn from the case's graph model, self loops as -1."""
    n, model = case["n"], case["model"]
    # ids are handed out with a little room: the last 1/256 of them have no edge yet
    n -= n // 256
    if model == "rmat":
        return gen.rmat_candidates(math.ceil(math.log2(n)), count, 0.57, 0.19, 0.19, g, DEV, n)
    if model == "chung_lu":
        cdf = torch.from_numpy(_chung_lu_cdf(n)).to(DEV)
        perm = torch.randperm(n, generator=_generator(g.initial_seed() + 1), device=DEV)  # hubs spread over the ids
        u, v = (perm[torch.searchsorted(cdf, torch.rand(count, generator=g, device=DEV, dtype=torch.float64))
                     .clamp_(max=n - 1)] for _ in range(2))
    elif model == "blocks":  # 64 blocks of consecutive ids, no edge between them
        size = -(-n // 64)
        u = torch.randint(0, n, (count,), generator=g, device=DEV)
        lo = u // size * size
        width = torch.clamp(n - lo, max=size)
        v = lo + (torch.rand(count, generator=g, device=DEV, dtype=torch.float64) * width).long().clamp_(max=size - 1)
        v = torch.minimum(v, lo + width - 1)
    else:
        u = torch.randint(0, n, (count,), generator=g, device=DEV)
        v = torch.randint(0, n, (count,), generator=g, device=DEV)
    key = (torch.minimum(u, v) << 32) | torch.maximum(u, v)
    key[u == v] = -1
    return key


def _edges(case, want, g):
    """`want` distinct edges of the case's model in random order (at most a quarter of all pairs)."""
    n = case["n"]
    want = min(want, n * (n // 64 if case["model"] == "blocks" else n - n // 128) // 8)
    keys = gen.first_occurrences(_candidates(case, int(want * 1.15) + 1024, g))
    while keys.numel() < want:
        more = _candidates(case, 4 * (want - keys.numel()) + 1024, g)
        keys = gen.first_occurrences(torch.cat([keys, more]))
    return keys[:want]


def _pairs(keys, g):
    """Edges as (src, dst) int32 pairs, either end first."""
    p = gen.keys_to_pairs(keys)
    swap = torch.rand(p.shape[0], generator=g, device=DEV) < 0.5
    return torch.where(swap[:, None], p.flip(1), p).contiguous()


def _base_and_churn(case, g):
    """The graph before the first pass, and a batch that deletes some of it and inserts as much."""
    keys = _edges(case, case["base"] + case["updates"] // 2, g)
    base = keys[: case["base"]]
    fresh = keys[base.numel():]
    gone = base[torch.randperm(base.numel(), generator=g, device=DEV)[: case["updates"] - fresh.numel()]]
    churn = torch.cat([gone, fresh])
    churn = churn[torch.randperm(churn.numel(), generator=g, device=DEV)]
    return _pairs(base, g), _pairs(churn, g)


def _config(case, **kw):
    return gz.CCAlgConfiguration(gamma_bytes=case["gamma"], **kw)


def _started(case, seed, base):
    """An instance that holds the base graph and has answered a query."""
    alg = gz.CCSketchAlg(case["n"], seed, _config(case))
    torch.cuda.synchronize()
    alg.ingest_pairs_device(base.data_ptr(), base.shape[0])
    alg.connected_components()
    return alg


def _tenant_sizes(case):
    lo, hi, count = case["log2_lo"], case["log2_hi"], case["tenants"]
    return [int(2.0 ** (lo + t / (count - 1) * (hi - lo))) for t in range(count)]


def prepare(case, seed):
    g = _generator(seed)
    rng = np.random.default_rng(seed)
    kind, n = case["kind"], case.get("n")
    if kind == "sketch":
        length = gz.calc_vector_length(n)
        s = gz.Sketch(length, seed, gz.calc_cc_samples(n), 1, case["gamma"])
        s.update_batch(rng.integers(0, length, 1000, dtype=np.uint64))
        if case["feed"] == "host":
            return dict(case=case, sketch=s, idx=rng.integers(0, length, case["count"], dtype=np.uint64))
        return dict(case=case, sketch=s, idx=torch.randint(0, length, (case["count"],), generator=g, device=DEV))
    if kind == "plugin":
        e = _edges(dict(model="uniform", n=n), n * case["per_vertex"] // 2, g)
        e = gen.keys_to_pairs(e).cpu().numpy().astype(np.uint32)
        half = e[: len(e) // 2]
        both = np.concatenate([e, e[:, ::-1]])
        both = both[np.argsort(both[:, 0], kind="stable")]
        cuts = np.flatnonzero(np.diff(both[:, 0])) + 1
        gutters = [(int(p[0, 0]), np.ascontiguousarray(p[:, 1])) for p in np.split(both, cuts)]
        alg = gz.CCSketchAlg(n, seed, _config(case, eager_dsu=False))
        alg.allocate_worker_memory(1)
        alg.ingest_pairs(half)
        alg.connected_components()
        return dict(case=case, alg=alg, gutters=gutters)
    if kind == "tenants":
        rows = []
        for t, m in enumerate(_tenant_sizes(case)):
            updates = int(case["per_nlogn"] * m * math.log2(m))
            pairs, _, _ = gen.rmat_stream(math.ceil(math.log2(m)), updates, 0.1, seed * 8 + t, DEV, n=m)
            rows.append((m, pairs))
        return dict(case=case, server=gz.Server(0, 4), pairs=[p for _, p in rows], ns=[m for m, _ in rows],
                    seeds=[seed + t for t in range(len(rows))], trace=gen.multi_tenant_trace(rows, 5, None))
    us = rng.integers(0, n, max(1, case.get("watch", 1)), dtype=np.uint32)
    fresh = rng.random(us.size) < 0.125  # one watched pair in eight is about an id without edges
    us[fresh] = n - 1 - rng.integers(0, max(1, n // 256), int(fresh.sum()), dtype=np.uint32)
    vs = rng.integers(0, n, us.size, dtype=np.uint32)
    if kind == "cached":
        base = _pairs(_edges(case, case["base"], g), g)
        alg = _started(case, seed, base)
        cc = alg.connected_components()
        ids, sizes = np.unique(cc.parent_arr, return_counts=True)
        giant = torch.from_numpy(np.flatnonzero(cc.parent_arr == ids[sizes.argmax()])).to(DEV)
        u, v = (giant[torch.randint(0, giant.numel(), (2 * case["updates"],), generator=g, device=DEV)] for _ in range(2))
        key = (torch.minimum(u, v) << 32) | torch.maximum(u, v)
        there = (torch.minimum(base[:, 0], base[:, 1]).long() << 32) | torch.maximum(base[:, 0], base[:, 1]).long()
        key[(u == v) | torch.isin(key, there)] = -1
        new = gen.first_occurrences(key)[: case["updates"]]
        return dict(case=case, alg=alg, batch=_pairs(new, g), us=us, vs=vs)
    base, churn = _base_and_churn(case, g)
    alg = _started(case, seed, base)
    if kind == "serve":
        # the arrival pattern belongs to the case and ends with one group of point queries; who asks
        # about whom comes from the seed, and one query in four is about an id without edges
        trace = gen.serving_trace(n, churn.shape[0], 5, case["per_request"], cc_frac=0.05)
        last = np.zeros(32, dtype=trace.dtype)
        last["kind"] = gz.REQ_POINT
        trace = np.concatenate([trace, last])
        point = trace["kind"] == gz.REQ_POINT
        trace["u"][point] = np.where(rng.random(point.sum()) < 0.25, n - 1, rng.integers(0, n - n // 256, point.sum()))
        trace["v"][point] = rng.integers(0, n - n // 256, point.sum())
        return dict(case=case, alg=alg, batch=churn, trace=trace)
    batch = churn.cpu().numpy().astype(np.uint32) if case["feed"] == "host" else churn
    return dict(case=case, alg=alg, batch=batch, us=us, vs=vs)


# ---- one pass ----------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sketch":
        s, idx = state["sketch"], state["idx"]
        s.reset_sample_state()
        if case["feed"] == "host":
            s.update_batch(idx)
        else:
            s.update_batch_device_noalloc(idx.data_ptr(), idx.numel())
        picked, code = s.sample()
        return {"sample": picked, "code": code, "image": np.frombuffer(s.serialize(), dtype=np.uint8)}
    if kind == "tenants":
        lat, answers, digests, stats = state["server"].run_trace(
            state["trace"], [p.data_ptr() for p in state["pairs"]], state["ns"], state["seeds"], _config(case))
        return {"answers": answers.astype(np.int64), "digests": digests.view(np.int64)}
    alg = state["alg"]
    if kind == "plugin":
        for src, dsts in state["gutters"]:
            alg.pre_insert(src, int(dsts[0]))  # without the eager DSU it only marks the answer as old
            alg.apply_update_batch(0, src, dsts)
        cc = alg.connected_components()
        return {"num_cc": cc.size(), "labels": cc.canonical_labels().astype(np.int64), "image": alg.dump_sketches()}
    if kind == "serve":
        lat, answers, stats = alg.serve_trace(state["batch"].data_ptr(), True, state["trace"])
        return {"answers": answers.astype(np.int64)}
    batch = state["batch"]
    if isinstance(batch, np.ndarray):
        alg.ingest_pairs(batch)
    else:
        alg.ingest_pairs_device(batch.data_ptr(), batch.shape[0])
    if kind == "cached" or case["ask"] == "points":
        return {"connected": alg.point_queries(state["us"], state["vs"])}
    cc = alg.connected_components()
    if case["ask"] == "labels":
        return {"num_cc": cc.size(), "labels": cc.canonical_labels().astype(np.int64)}
    return {"num_cc": cc.size(), "connected": alg.point_queries(state["us"], state["vs"])}


# ---- what a pass cannot do without -------------------------------------------------------------
def _geometry(n, gamma):
    c, d = gz.calc_cc_samples(n), gz.calc_bkt_per_col(gz.calc_vector_length(n))
    rec = 8 + gamma
    return c, d, rec, (c * d + 1) * rec


def _ingest_bytes(n, updates, gamma):
    """The pairs read once, and every bucket an update toggles read and written once (a vertex's
    sketch at most whole)."""
    c, d, rec, sketch = _geometry(n, gamma)
    per_vertex = 2 * updates / n
    touched = min(sketch, per_vertex * (c + 1) * rec) * n if per_vertex >= 1 else 2 * updates * (c + 1) * rec
    return 8 * updates + 2 * touched


def _query_bytes(n, gamma):
    """One column and the deterministic bucket of every vertex, and its root written."""
    c, d, rec, sketch = _geometry(n, gamma)
    return n * ((d + 1) * rec + 4)


def work(case):
    kind, gamma = case["kind"], case["gamma"]
    if kind == "sketch":
        return {"bytes": 8 * case["count"] + 2 * _geometry(case["n"], gamma)[3], "flops": 0}
    if kind == "tenants":
        total = 0.0
        for n in _tenant_sizes(case):
            total += _ingest_bytes(n, case["per_nlogn"] * n * math.log2(n), gamma) + 9 * _query_bytes(n, gamma)
        return {"bytes": total, "flops": 0}
    n = case["n"]
    if kind == "plugin":
        return {"bytes": _ingest_bytes(n, n * case["per_vertex"] // 2, gamma) + _query_bytes(n, gamma)
                + 2 * n * _geometry(n, gamma)[3], "flops": 0}
    if kind == "cached":  # the pairs read, both ends' roots read, the pairs kept for the next flush
        return {"bytes": 24 * case["updates"] + 17 * case["watch"], "flops": 0}
    if kind == "serve":
        groups = max(1, case["updates"] // max(case["per_request"], 150_000))
        return {"bytes": groups * (_ingest_bytes(n, case["updates"] // groups, gamma) + _query_bytes(n, gamma)),
                "flops": 0}
    return {"bytes": _ingest_bytes(n, case["updates"], gamma) + _query_bytes(n, gamma) + 9 * case["watch"], "flops": 0}
