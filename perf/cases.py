"""Performance cases of the framework: what a GNN training job has it do, through its public entry points.

A job keeps node features and the graph's adjacency in pinned host memory and the hot part of both in HBM. It builds
the maps and the cached sub-graph when its cache is (re)made, and then, batch after batch, samples neighbours, relabels
ids and fetches feature rows; learnable features are written back with cache_set. The cases run these calls on
synthetic graphs and tables of the sizes that bench.py and the tests use, from a few rows to a whole mini-batch.
"""
import math

import torch

import shmtensor_amd
from shmtensor_amd.synthetic import rmat_csr, zipf_ranks

capi = shmtensor_amd.install_aliases()
from shmtensor_amd.shmtensor import GPUSamplingDataloader  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i64": torch.int64}


def listed():
    return [
        # A serving-style lookup of a handful of nodes; 90 % of the table cached under random ids. Latency only.
        dict(name="fetch_few", kind="fetch", rows=200_000, dim=128, dtype="f32", cached=0.9, skew=False, queries=64,
             id_bytes=8, layout="auto"),
        # The small fetch benchmark: a quarter of the rows is cached, so the host link carries most of the batch.
        dict(name="fetch_quarter_cached", kind="fetch", rows=200_000, dim=128, dtype="f32", cached=0.25, skew=False,
             queries=65_536, id_bytes=8, layout="auto"),
        # A large skewed batch through the general table: hot ids repeat, a few per cent of the rows miss.
        dict(name="fetch_zipf_large", kind="fetch", rows=16_000_000, dim=128, dtype="f16", cached=0.4, skew=True,
             queries=1_048_576, id_bytes=8, layout="buckets"),
        # Write-back of one step's updated embedding rows; 100 floats a row (400 bytes, no power of two), all cached.
        dict(name="set_rows", kind="set", rows=1_000_000, dim=100, dtype="f32", cached=1.0, updates=262_144, id_bytes=8,
             layout="auto"),
        # The static map made from scratch for 4 M sparse 40-bit keys, and the first batch looked up in it.
        dict(name="map_build", kind="map_build", keys=4_194_304, key_bits=40, id_bytes=8, load_factor=0.5,
             queries=524_288),
        # A bulk lookup in that map: half of the requests are keys, half are not.
        dict(name="map_query", kind="map_query", keys=4_194_304, key_bits=40, id_bytes=8, load_factor=0.5,
             queries=16_777_216),
        # One sampling hop over a CSR whose rows of the highest degree (30 %) are cached; the rest is read over the link.
        dict(name="sample_cached", kind="sample", rows=400_000, max_degree=1000, cached=0.3, seeds=100_000, fanout=5,
             replace=False, index_bytes=4),
        # The cached sub-graph copied out of pinned host memory when the cache is made.
        dict(name="subcsr", kind="subcsr", rows=400_000, max_degree=1000, cached=0.3, index_bytes=4),
        # The seeds and sampled ids of a large hop mapped to dense labels, hub nodes repeating as they do in real graphs.
        dict(name="relabel_large", kind="relabel", seeds=130_000, ids=3_000_000, nodes=2_000_000, id_bytes=4),
        # A training epoch's sampling, one batch at a time: latency of the chain of hops.
        dict(name="loader_single", kind="loader", scale=21, edge_factor=30, cached=0.3, batch=1024, batches=4,
             fanouts="15,10,5", prefetch=1, dim=0, rows_cached=0.0),
        # The same with eight batches sampled together (prefetch), launches shared between them.
        dict(name="loader_prefetch", kind="loader", scale=21, edge_factor=30, cached=0.3, batch=1024, batches=8,
             fanouts="15,10,5", prefetch=8, dim=0, rows_cached=0.0),
        # Whole mini-batches: three hops and the feature rows of all input nodes, pipelined over the host link.
        dict(name="loader_features", kind="loader", scale=22, edge_factor=16, cached=0.2, batch=4096, batches=4,
             fanouts="25,15,10", prefetch=4, dim=256, rows_cached=0.25),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fetch", "fetch", "set", "map_build", "map_query", "sample", "subcsr", "relabel", "loader", "loader"])
    if kind == "fetch" or kind == "set":
        dim, dtype = rng.choice([1, 16, 33, 50, 64, 100, 128, 200, 256, 300]), rng.choice(sorted(DTYPES))
        row_bytes = dim * torch.empty(0, dtype=DTYPES[dtype]).element_size()
        most = min(16_000_000, (1 << 31) // row_bytes)
        rows = _log_int(rng, 20_000, most if kind == "fetch" else min(most, 1_000_000))
        c = dict(kind=kind, rows=rows, dim=dim, dtype=dtype, id_bytes=rng.choice([4, 8]),
                 layout=rng.choice(["auto", "auto", "buckets"]))
        if kind == "fetch":
            # (the link carries what misses: at most 64 MB of it)
            cached = rng.choice([0.25, 0.5, 0.9, 1.0])
            most = min(1_048_576, (1 << 26) / (row_bytes * (1.0 - cached)) if cached < 1.0 else 1 << 20)
            return dict(c, cached=cached, skew=rng.random() < 0.5, queries=_log_int(rng, 16, most))
        return dict(c, cached=1.0, updates=_log_int(rng, 16, min(rows, 262_144)))
    if kind == "map_build":
        id_bytes = rng.choice([4, 8])
        return dict(kind=kind, keys=_log_int(rng, 1_000, 4_194_304), key_bits=rng.choice([24, 30] if id_bytes == 4 else [24, 30, 40]),
                    id_bytes=id_bytes, load_factor=rng.choice([0.3, 0.5, 0.8]), queries=524_288)
    if kind == "map_query":
        id_bytes = rng.choice([4, 8])
        return dict(kind=kind, keys=_log_int(rng, 1_000, 4_194_304), key_bits=rng.choice([24, 30] if id_bytes == 4 else [24, 30, 40]),
                    id_bytes=id_bytes, load_factor=rng.choice([0.3, 0.5, 0.8]), queries=_log_int(rng, 1_000, 16_777_216))
    if kind == "sample":
        rows = _log_int(rng, 10_000, 400_000)
        return dict(kind=kind, rows=rows, max_degree=rng.choice([20, 100, 300, 1000]), cached=rng.choice([0.0, 0.3, 0.3, 1.0]),
                    seeds=_log_int(rng, 10, min(rows, 100_000)), fanout=rng.choice([3, 5, 10, 15, 25, 40]),
                    replace=rng.random() < 0.3, index_bytes=rng.choice([4, 8]))
    if kind == "subcsr":
        return dict(kind=kind, rows=_log_int(rng, 10_000, 400_000), max_degree=rng.choice([20, 100, 300, 1000]),
                    cached=rng.choice([0.1, 0.2, 0.3]), index_bytes=rng.choice([4, 8]))
    if kind == "relabel":
        ids = _log_int(rng, 1_000, 16_000_000)
        return dict(kind=kind, seeds=max(1, ids // rng.choice([5, 10, 25])), ids=ids,
                    nodes=max(1000, int(ids * rng.uniform(0.2, 2.0))), id_bytes=rng.choice([4, 8]))
    dim = rng.choice([0, 0, 64, 100, 128])
    batches = rng.randint(1, 8 if dim == 0 else 4)
    return dict(kind="loader", scale=rng.randint(15, 21), edge_factor=rng.choice([8, 16, 30]), cached=rng.choice([0.1, 0.2, 0.3]),
                batch=_log_int(rng, 64, 1024), batches=batches, fanouts=rng.choice(["15,10,5", "25,10", "10,10", "5,5,5", "20,15,10"]),
                prefetch=rng.choice([1, 4, 8]), dim=dim, rows_cached=rng.choice([0.25, 0.5]) if dim else 0.0)


def _ids(t, nbytes):
    return t.to(torch.int32 if nbytes == 4 else torch.int64)


def _pinned(t):
    return torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t)


def _unique_keys(n, bits, g):
    """n distinct ids of [0, 2^bits) in random order."""
    if bits <= 24:
        return torch.randperm(1 << bits, device="cuda", generator=g)[:n].contiguous()
    pool = torch.unique(torch.randint(0, 1 << bits, (n + n // 8 + 64,), device="cuda", generator=g))
    return pool[torch.randperm(pool.numel(), device="cuda", generator=g)[:n]].contiguous()


def _random_rows(rows, dim, dtype, g):
    if dtype == torch.int64:
        return torch.randint(-(1 << 40), 1 << 40, (rows, dim), device="cuda", generator=g)
    return torch.randn((rows, dim), device="cuda", generator=g, dtype=torch.float32).to(dtype)


def _feature_state(case, g):
    """The id-addressed table in pinned host memory, the cached rows in HBM (hottest first, under scattered ids), their
    map, and the ids by hotness."""
    rows = case["rows"]
    table_dev = _random_rows(rows, case["dim"], DTYPES[case["dtype"]], g)
    by_heat = torch.randperm(rows, device="cuda", generator=g)
    hot = by_heat[: max(1, int(rows * case["cached"]))]
    table, cache = _pinned(table_dev), table_dev[hot]
    hmap = capi.CUCOStaticHashmap(_ids(hot, case["id_bytes"]), _ids(torch.arange(hot.numel(), device="cuda"), case["id_bytes"]),
                                  0.8, layout=case["layout"])
    return table, cache, hmap, by_heat


# Results have data-dependent sizes (edges of a sample, distinct ids). What decides these sizes is the same for every seed
# of a case, so that the outputs of two seeds have one shape; what they hold differs: ids, neighbours, order, values.

def _uniform_csr(case, g):
    """A CSR of rows with degrees uniform in [0, max_degree) (the same for every seed) and random neighbours, and the ids
    of its rows of the highest degree that are cached, in id order."""
    rows, index = case["rows"], torch.int32 if case["index_bytes"] == 4 else torch.int64
    fixed = torch.Generator(device="cuda").manual_seed(rows + case["max_degree"])
    deg = torch.randint(0, case["max_degree"], (rows,), device="cuda", generator=fixed)
    indptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(deg, 0, out=indptr[1:])
    indices = torch.randint(0, rows, (int(indptr[-1]),), device="cuda", generator=g, dtype=index)
    top = torch.sort(deg, descending=True, stable=True).indices[: int(rows * case["cached"])]
    return indptr, indices, torch.sort(top).values.contiguous()


def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "fetch":
        table, cache, hmap, by_heat = _feature_state(case, g)
        if case["skew"]:
            q = by_heat[zipf_ranks(case["queries"], case["rows"], 1.1, seed=seed + 1)]
        else:
            q = torch.randint(0, case["rows"], (case["queries"],), device="cuda", generator=g)
        return dict(kind=kind, args=(table, cache, _ids(q, case["id_bytes"]).contiguous(), hmap))
    if kind == "set":
        table, cache, hmap, _ = _feature_state(case, g)
        q = torch.randperm(case["rows"], device="cuda", generator=g)[: case["updates"]]
        update = _random_rows(case["updates"], case["dim"], DTYPES[case["dtype"]], g)
        return dict(kind=kind, args=(table, cache, _ids(q, case["id_bytes"]).contiguous(), update, hmap))
    if kind in ("map_build", "map_query"):
        keys = _unique_keys(case["keys"], case["key_bits"], g)
        n, nq = keys.numel(), case["queries"]
        members = keys[torch.randint(0, n, ((nq + 1) // 2,), device="cuda", generator=g)]
        others = torch.randint(0, 1 << case["key_bits"], (nq // 2,), device="cuda", generator=g)   # (hardly ever keys)
        q = torch.cat([members, others])[torch.randperm(nq, device="cuda", generator=g)]
        keys, q = _ids(keys, case["id_bytes"]).contiguous(), _ids(q, case["id_bytes"]).contiguous()
        values = _ids(torch.arange(n, device="cuda"), case["id_bytes"])
        if kind == "map_build":
            return dict(kind=kind, keys=keys, values=values, load_factor=case["load_factor"], requests=q)
        return dict(kind=kind, map=capi.CUCOStaticHashmap(keys, values, case["load_factor"]), requests=q)
    if kind == "sample":
        indptr, indices, top = _uniform_csr(case, g)
        fixed = torch.Generator(device="cuda").manual_seed(case["seeds"])
        seeds = torch.randperm(case["rows"], device="cuda", generator=fixed)[: case["seeds"]]
        seeds = seeds[torch.randperm(case["seeds"], device="cuda", generator=g)].contiguous()
        more = dict(seeds=seeds, fanout=case["fanout"], replace=case["replace"], rng=seed)
        if case["cached"] >= 1.0:
            return dict(kind=kind, csr=(indptr, indices), cached=None, **more)
        csr = (_pinned(indptr), _pinned(indices))
        if top.numel() == 0:
            return dict(kind=kind, csr=csr, cached=None, **more)
        sub = capi.create_subcsr(csr[0], csr[1], top)
        hmap = capi.CUCOStaticHashmap(top, torch.arange(top.numel(), device="cuda"), 0.8)
        return dict(kind=kind, csr=csr, cached=(sub[0], sub[1], hmap), **more)
    if kind == "subcsr":
        indptr, indices, top = _uniform_csr(case, g)
        return dict(kind=kind, args=(_pinned(indptr), _pinned(indices), top))
    if kind == "relabel":
        nodes = case["nodes"]
        name = torch.randperm(nodes, device="cuda", generator=g)         # (hot nodes have any id)
        fixed = torch.Generator(device="cuda").manual_seed(case["ids"])
        seeds = torch.randint(0, nodes, (case["seeds"],), device="cuda", generator=fixed)
        heat = torch.rand(case["ids"], device="cuda", generator=fixed, dtype=torch.float64).pow_(2.5)
        ids = (heat * nodes).to(torch.int64).clamp_(max=nodes - 1)
        seeds = name[seeds[torch.randperm(case["seeds"], device="cuda", generator=g)]]
        ids = name[ids[torch.randperm(case["ids"], device="cuda", generator=g)]]
        return dict(kind=kind, tensors=[_ids(seeds, case["id_bytes"]).contiguous(), _ids(ids, case["id_bytes"]).contiguous()])
    # a dataloader over an R-MAT graph: adjacency of the nodes of the highest degree cached in HBM
    # (graph, batches and random base are the same for every seed; the order of each batch's nodes and the feature rows
    # differ: a node's sample does not depend on its place in the batch, so the sizes of the results do not either)
    indptr_dev, indices_dev = rmat_csr(case["scale"], case["edge_factor"], seed=case["scale"])
    n = indptr_dev.numel() - 1
    deg = indptr_dev[1:] - indptr_dev[:-1]
    by_degree = torch.sort(deg, descending=True, stable=True).indices
    hot = torch.sort(by_degree[: int(n * case["cached"])]).values.contiguous()
    indptr, indices = _pinned(indptr_dev), _pinned(indices_dev)
    features = None
    if case["dim"]:
        rows_dev = _random_rows(n, case["dim"], torch.float32, g)
        kept = torch.sort(by_degree[: int(n * case["rows_cached"])]).values
        features = (_pinned(rows_dev), rows_dev[kept],
                    capi.CUCOStaticHashmap(kept, torch.arange(kept.numel(), device="cuda"), 0.8))
    fixed = torch.Generator(device="cuda").manual_seed(case["batch"])
    seeds = torch.randperm(n, device="cuda", generator=fixed)[: case["batch"] * case["batches"]].view(case["batches"], -1)
    order = torch.rand(seeds.shape, device="cuda", generator=g).argsort(dim=1)
    seeds = torch.gather(seeds, 1, order).flatten()
    loader = GPUSamplingDataloader(indptr, indices, seeds, case["batch"], [int(k) for k in case["fanouts"].split(",")],
                                   shuffle=False, rng_seed=7777, prefetch=case["prefetch"], features=features)
    loader.gpu_indptr, loader.gpu_indices = capi.create_subcsr(indptr, indices, hot)
    loader.hashmap = capi.CUCOStaticHashmap(hot, torch.arange(hot.numel(), device="cuda"), 0.8)
    loader.has_cache = True
    return dict(kind=kind, loader=loader)


def run(state):
    kind = state["kind"]
    if kind == "fetch":
        return capi.cache_fetch(*state["args"])
    if kind == "set":
        capi.cache_set(*state["args"])
        return state["args"][1]
    if kind == "map_build":
        return capi.CUCOStaticHashmap(state["keys"], state["values"], state["load_factor"]).query(state["requests"])
    if kind == "map_query":
        return state["map"].query(state["requests"])
    if kind == "sample":
        if state["cached"] is None:
            return capi.csr_sampling(*state["csr"], state["seeds"], state["fanout"], state["replace"], seed=state["rng"])
        return capi.csr_cache_sampling(*state["csr"], *state["cached"], state["seeds"], state["fanout"], state["replace"],
                                       seed=state["rng"])
    if kind == "subcsr":
        return capi.create_subcsr(*state["args"])
    if kind == "relabel":
        return capi.tensor_relabel(state["tensors"])
    # one epoch; every batch is what a training step is handed: input nodes, the blocks' edges, the feature rows
    return [[batch[0], [(b.indptr, b.indices) for b in batch[2]], list(batch[3:])] for batch in state["loader"]]


def work(case):
    kind = case["kind"]
    if kind in ("fetch", "set"):
        row_bytes = case["dim"] * torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
        moved = case["queries"] if kind == "fetch" else case["updates"]
        return {"bytes": moved * (2 * row_bytes + case["id_bytes"]), "flops": 0}
    if kind in ("map_build", "map_query"):
        # building reads every pair and writes it once into a slot; a lookup reads its request and a slot, writes a value
        build = 4 * case["keys"] * case["id_bytes"] if kind == "map_build" else 0
        return {"bytes": build + 4 * case["queries"] * case["id_bytes"], "flops": 0}
    if kind == "sample":
        # per seed its id, two row offsets and the output offset; per edge the neighbour read and written
        edges = case["seeds"] * _mean_picks(case)
        return {"bytes": case["seeds"] * (8 + 16 + 8) + edges * 2 * case["index_bytes"], "flops": 0}
    if kind == "subcsr":
        c = case["cached"]
        edges = case["rows"] * c * case["max_degree"] * (1 - c / 2)
        return {"bytes": case["rows"] * c * (8 + 16 + 8) + edges * 2 * case["index_bytes"], "flops": 0}
    if kind == "relabel":
        n = case["seeds"] + case["ids"]
        return {"bytes": n * 2 * case["id_bytes"] + 0.5 * case["nodes"] * case["id_bytes"], "flops": 0}
    # per hop and seed: its id, two row offsets, the output offset; per edge: the neighbour read, its label written;
    # then the unique ids, and the feature rows read and written
    # (how many picks a node has and how many distinct nodes they are was counted on R-MAT graphs: half of the nodes a
    # batch starts from have hardly a neighbour, and the hubs are met again and again)
    total, frontier, reached = 0.0, float(case["batch"]), 0.1 * (1 << case["scale"])
    for k, filled in zip(reversed([int(k) for k in case["fanouts"].split(",")]), (0.45, 0.8, 0.93)):
        edges = filled * frontier * k
        total += frontier * (8 + 16 + 8) + edges * (4 + 8)
        frontier = reached * (1.0 - math.exp(-(frontier + edges) / reached))
        total += frontier * 8
    total += frontier * 2 * case["dim"] * 4
    return {"bytes": total * case["batches"], "flops": 0}


def _mean_picks(case):
    """Mean picks of a row whose degree is uniform in [0, max_degree)."""
    d, k = case["max_degree"], case["fanout"]
    if case["replace"]:
        return k * (1 - 1 / d)
    return k if d <= 1 else sum(min(k, i) for i in range(d)) / d


def tolerance(case):
    # ids, labels and values are whole numbers and rows are moved as bytes; samples are a function of the given seed
    return "exact"
