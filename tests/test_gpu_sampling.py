"""Neighbour sampling and the cached sub-CSR on the GPU: the reference's
known-answer cases (example/test_cache_sampling.py:23-126), the CPU oracle,
structural invariants, and chi-square tests of the uniform law."""
import numpy as np
import pytest
import torch
from scipy.stats import chi2 as chi2_dist

from conftest import load_golden

pytestmark = pytest.mark.gpu


def _kat_check(g, sp, si, replace):
    exp = g["replace_true" if replace else "replace_false"]
    assert sp.tolist() == exp["sub_indptr"]
    assert si.numel() == exp["sub_indptr"][-1]
    seg = lambda i: si[sp[i]:sp[i + 1]]
    if replace:
        for i, (lo, hi) in enumerate(exp["segment_ranges"]):
            assert bool(((seg(i) >= lo) & (seg(i) < hi)).all())
    else:
        for i, vals in exp["exact_segments"].items():
            assert seg(int(i)).tolist() == vals
        for i, (lo, hi) in exp["distinct_in_range"].items():
            s = seg(int(i))
            assert bool(((s >= lo) & (s < hi)).all()) and s.unique().numel() == g["num_picks"]


@pytest.mark.parametrize("replace", [True, False])
def test_csr_sampling_reference_kat(capi, replace):
    g = load_golden("csr_sampling_kat.json")
    indptr = torch.tensor(g["indptr"]).long().cuda()
    indices = torch.arange(g["num_indices"]).long().cuda()
    seeds = torch.tensor(g["seeds"]).int().cuda()
    sp, si = capi.csr_sampling(indptr, indices, seeds, g["num_picks"], replace)
    assert sp.dtype == torch.int64 and si.dtype == torch.int64 and sp.is_cuda and si.is_cuda
    _kat_check(g, sp, si, replace)
    again = capi.csr_sampling(indptr, indices, seeds, g["num_picks"], replace)
    assert torch.equal(again[1], si)          # fixed default seed: same call, same sample


def test_csr_cache_sampling_reference_kat(capi):
    g = load_golden("csr_sampling_kat.json")
    s = load_golden("subcsr_kat.json")
    indptr = torch.tensor(g["indptr"]).long().pin_memory()
    indices = torch.arange(g["num_indices"]).long().pin_memory()
    capi.pin_memory(indptr)
    capi.pin_memory(indices)
    cache_seeds = torch.tensor(g["cache_seeds"]).long().cuda()
    gp, gi = capi.create_subcsr(indptr, indices, cache_seeds)
    assert gp.tolist() == s["gpu_indptr"] and gi.tolist() == s["gpu_indices"]
    h = capi.CUCOStaticHashmap(cache_seeds, torch.arange(cache_seeds.numel()).cuda().long(), 0.8)
    seeds = torch.tensor(g["seeds"]).int().cuda()          # int32 seeds against int64 keys
    for replace in (True, False):
        sp, si = capi.csr_cache_sampling(indptr, indices, gp, gi, h, seeds, g["num_picks"], replace)
        _kat_check(g, sp, si, replace)
    capi.unpin_memory(indptr)
    capi.unpin_memory(indices)


def _random_csr(rng, n, max_deg, ptr_dt, idx_dt, hubs=()):
    deg = rng.integers(0, max_deg, size=n)
    deg[rng.integers(0, n, size=n // 10)] = 0
    for v, d in hubs:
        deg[v] = d
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(ptr_dt)
    indices = rng.integers(0, n, size=int(indptr[-1])).astype(idx_dt)
    return indptr, indices


@pytest.mark.parametrize("ptr_dt,idx_dt", [(np.int64, np.int64), (np.int32, np.int32), (np.int64, np.int32)])
@pytest.mark.parametrize("seed_dt", [np.int32, np.int64])
@pytest.mark.parametrize("k", [1, 5, 10, 15, 25, 64, 65, 200])
def test_sampling_matches_oracle_bit_exact(capi, oracle, ptr_dt, idx_dt, seed_dt, k):
    """Uncached and cached sampling against the oracle: sub_indptr and every
    deg <= k segment follow the reference rules; deg > k segments equal the
    oracle's restatement of the device selection rule (Floyd + Philox), which
    in turn is checked for uniformity in tests/test_oracle.py."""
    rng = np.random.default_rng(k * 131 + np.dtype(ptr_dt).itemsize + np.dtype(seed_dt).itemsize)
    n = 4000
    indptr, indices = _random_csr(rng, n, 40, ptr_dt, idx_dt, hubs=[(7, 5000), (8, k), (9, k + 1), (10, 300)])
    seeds = np.concatenate([[7, 8, 9, 10, 7], rng.integers(0, n, size=5001)]).astype(seed_dt)
    t = lambda a: torch.from_numpy(a)
    hp, hx = t(indptr).pin_memory(), t(indices).pin_memory()
    for replace in (False, True):
        esp, esi = oracle.sample(indptr, indices, seeds, k, replace, seed=7777, algo="floyd")
        sp, si = capi.csr_sampling(hp, hx, t(seeds).cuda(), k, replace)
        assert sp.dtype == t(indptr).dtype and si.dtype == t(indices).dtype
        assert np.array_equal(sp.cpu().numpy(), esp)
        assert np.array_equal(si.cpu().numpy(), esi)
        sp2, si2 = capi.csr_sampling(hp.cuda(), hx.cuda(), t(seeds).cuda(), k, replace)   # fully on the GPU
        assert torch.equal(sp2, sp) and torch.equal(si2, si)
    # cache the 30 % highest-degree rows; the result must not change
    order = np.argsort(-(indptr[1:] - indptr[:-1]), kind="stable")[: n * 3 // 10].astype(np.int64)
    gp, gi = capi.create_subcsr(hp, hx, t(order).cuda())
    egp, egi = oracle.create_subcsr(indptr, indices, order)
    assert np.array_equal(gp.cpu().numpy(), egp) and np.array_equal(gi.cpu().numpy(), egi)
    for key_dt in (torch.int32, torch.int64):
        h = capi.CUCOStaticHashmap(t(order).to(key_dt).cuda(), torch.arange(order.size, dtype=key_dt).cuda(), 0.8)
        sp3, si3 = capi.csr_cache_sampling(hp, hx, gp, gi, h, t(seeds).cuda(), k, False)
        esp, esi = oracle.sample(indptr, indices, seeds, k, False, seed=7777, algo="floyd")
        assert np.array_equal(sp3.cpu().numpy(), esp) and np.array_equal(si3.cpu().numpy(), esi)


def test_sampling_invariants_large_batch(capi, oracle):
    """S large enough for the multi-workgroup plan; every output is a true
    neighbour, no duplicates within a segment, exactly min(k, deg) per seed."""
    rng = np.random.default_rng(77)
    n, k = 200_000, 10
    indptr, indices_dup = _random_csr(rng, n, 60, np.int64, np.int32)
    # distinct neighbours per row so that "no duplicates" is meaningful
    indices = np.concatenate([rng.choice(n, size=d, replace=False) for d in np.diff(indptr[:2001])] +
                             [np.arange(indptr[2000], indptr[-1]) % n]).astype(np.int32)
    seeds = rng.permutation(n)[:150_000].astype(np.int64)
    hp, hx = torch.from_numpy(indptr).pin_memory(), torch.from_numpy(indices).pin_memory()
    sp, si = capi.csr_sampling(hp, hx, torch.from_numpy(seeds).cuda(), k, False, seed=123)
    deg = (indptr[1:] - indptr[:-1])[seeds]
    assert np.array_equal(np.diff(sp.cpu().numpy()), np.minimum(deg, k))
    esp, esi = oracle.sample(indptr, indices, seeds, k, False, seed=123, algo="floyd")
    assert np.array_equal(si.cpu().numpy(), esi)
    sp_n, si_n = sp.cpu().numpy(), si.cpu().numpy()
    for s in range(0, 150_000, 997):
        seg = si_n[sp_n[s]:sp_n[s + 1]]
        adj = indices[indptr[seeds[s]]:indptr[seeds[s] + 1]]
        assert np.isin(seg, adj).all()
        if seeds[s] < 2000:
            assert np.unique(seg).size == seg.size


@pytest.mark.parametrize("deg,k", [(6, 5), (12, 5), (100, 15), (1000, 25), (70, 65)])
def test_uniform_without_replacement_chi_square(capi, deg, k):
    """Per-edge selection frequency over many independent seeds: each of the deg
    neighbours must be chosen with probability k/deg (df = deg-1, level 1e-6)."""
    trials = 40_000
    indptr = torch.arange(0, (trials + 1) * deg, deg)
    indices = torch.arange(deg).repeat(trials).int()
    sp, si = capi.csr_sampling(indptr.cuda(), indices.cuda(), torch.arange(trials).cuda(), k, False, seed=2024)
    assert torch.equal(sp.cpu(), torch.arange(trials + 1) * k)
    picks = si.view(trials, k)
    assert bool((picks.sort(dim=1).values.diff(dim=1) > 0).all())        # distinct within every segment
    counts = torch.bincount(si.long(), minlength=deg).cpu().numpy()
    expected = trials * k / deg
    stat = ((counts - expected) ** 2 / expected).sum() / (1 - k / deg)
    assert stat < chi2_dist.ppf(1 - 1e-6, deg - 1), (stat, counts)
    # a different seed or stream id gives a different sample
    _, si2 = capi.csr_sampling(indptr.cuda(), indices.cuda(), torch.arange(trials).cuda(), k, False, seed=2025)
    _, si3 = capi.csr_sampling(indptr.cuda(), indices.cuda(), torch.arange(trials).cuda(), k, False, seed=2024,
                               stream_id=1)
    assert not torch.equal(si, si2) and not torch.equal(si, si3)


def test_uniform_with_replacement_chi_square(capi):
    deg, k, trials = 9, 4, 40_000
    indptr = torch.arange(0, (trials + 1) * deg, deg)
    indices = torch.arange(deg).repeat(trials)
    _, si = capi.csr_sampling(indptr.cuda(), indices.cuda(), torch.arange(trials).cuda(), k, True, seed=1)
    counts = torch.bincount(si, minlength=deg).cpu().numpy()
    expected = trials * k / deg
    assert ((counts - expected) ** 2 / expected).sum() < chi2_dist.ppf(1 - 1e-6, deg - 1)


def test_empty_and_degenerate(capi):
    indptr = torch.tensor([0, 0, 3]).cuda()
    indices = torch.tensor([5, 6, 7]).int().cuda()
    sp, si = capi.csr_sampling(indptr, indices, torch.zeros(0, dtype=torch.int64).cuda(), 5, False)
    assert sp.tolist() == [0] and si.numel() == 0 and si.dtype == torch.int32
    sp, si = capi.csr_sampling(indptr, indices, torch.tensor([0, 0]).cuda(), 5, False)
    assert sp.tolist() == [0, 0, 0] and si.numel() == 0
    sp, si = capi.csr_sampling(indptr, indices, torch.tensor([1, 1]).cuda(), 0, False)
    assert sp.tolist() == [0, 0, 0] and si.numel() == 0
    sp, si = capi.csr_sampling(indptr, indices, torch.tensor([1, 0, 1]).cuda(), 1 << 40, False)   # "take all"
    assert sp.tolist() == [0, 3, 3, 6] and si.tolist() == [5, 6, 7, 5, 6, 7]
    gp, gi = capi.create_subcsr(indptr, indices, torch.zeros(0, dtype=torch.int64).cuda())
    assert gp.tolist() == [0] and gi.numel() == 0


def test_rmat_three_hop_pipeline(capi, oracle):
    """Config-3 shape at reduced scale (R-MAT scale 16, edge factor 30): top 30 %
    of rows by degree cached, 1,024 seeds, fanouts [15, 10, 5] applied in the
    dataloader's order (python/shmtensor/sampling.py:128), relabel after each hop.
    Checked hop by hop against the oracle pipeline."""
    from shmtensor_amd.synthetic import rmat_csr
    indptr_d, indices_d = rmat_csr(16, 30, seed=1)
    n = indptr_d.numel() - 1
    indptr, indices = indptr_d.cpu().pin_memory(), indices_d.cpu().pin_memory()
    deg = indptr[1:] - indptr[:-1]
    hot = torch.sort(deg, descending=True, stable=True).indices[: n * 3 // 10].cuda()
    gp, gi = capi.create_subcsr(indptr, indices, hot)
    h = capi.CUCOStaticHashmap(hot, torch.arange(hot.numel()).cuda(), 0.8)
    ref_cache = (gp.cpu().numpy(), gi.cpu().numpy(), oracle.Hashmap(hot.cpu().numpy(), np.arange(hot.numel()), 0.8))
    g = torch.Generator().manual_seed(4)
    seeds = torch.randperm(n, generator=g)[:1024].cuda()
    ref_seeds = seeds.cpu().numpy()
    total_edges = 0
    for hop, k in enumerate(reversed([15, 10, 5])):
        sp, si = capi.csr_cache_sampling(indptr, indices, gp, gi, h, seeds, k, False, stream_id=hop)
        u, (ls, ln) = capi.tensor_relabel([seeds, si])
        esp, esi = oracle.sample(indptr.numpy(), indices.numpy(), ref_seeds, k, False, cache=ref_cache,
                                 seed=7777, stream=hop, algo="floyd")
        eu, (els, eln) = oracle.relabel([ref_seeds, esi])
        assert np.array_equal(sp.cpu().numpy(), esp) and np.array_equal(si.cpu().numpy(), esi)
        assert np.array_equal(u.cpu().numpy(), eu) and np.array_equal(ln.cpu().numpy(), eln)
        assert torch.equal(u[: seeds.numel()], seeds)
        total_edges += si.numel()
        seeds, ref_seeds = u, eu
    assert total_edges > 50_000


def test_config3_full_size_properties(capi):
    """Configuration 3 at full size (R-MAT scale 21, 116 M edges, top 30 % of rows cached, 1,024 seeds,
    fanouts [15, 10, 5] in the dataloader's order): properties that need no CPU pass over the graph.
    Counts are min(k, degree); every sampled id is a neighbour of its seed, without repeats; the cache is
    transparent; the fused hop equals the separate operators; relabel inverts and keeps the seeds first."""
    from shmtensor_amd.synthetic import rmat_csr
    indptr_d, indices_d = rmat_csr(21, 30, seed=1)
    n = indptr_d.numel() - 1
    indptr, indices = indptr_d.cpu().pin_memory(), indices_d.cpu().pin_memory()
    deg = indptr_d[1:] - indptr_d[:-1]
    hot = torch.sort(deg, descending=True, stable=True).indices[: n * 3 // 10].contiguous()
    gp, gi = capi.create_subcsr(indptr, indices, hot)
    h = capi.CUCOStaticHashmap(hot, torch.arange(hot.numel(), device="cuda"), 0.8)
    # every edge as one sorted key (rows ascending, neighbours sorted within a row)
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    edge_keys = rows * n + indices_d.long()
    del rows
    seeds = torch.randperm(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(33))[:1024]
    for hop, k in enumerate([5, 10, 15]):
        sp, si = capi.csr_cache_sampling(indptr, indices, gp, gi, h, seeds, k, False, seed=7777, stream_id=hop)
        assert torch.equal(sp[1:] - sp[:-1], torch.clamp(deg[seeds], max=k))
        owner = torch.repeat_interleave(seeds, sp[1:] - sp[:-1])
        keys = owner * n + si.long()
        pos = torch.searchsorted(edge_keys, keys)
        assert bool((edge_keys[pos.clamp(max=edge_keys.numel() - 1)] == keys).all())      # real neighbours
        slot = torch.repeat_interleave(torch.arange(seeds.numel(), device="cuda"), sp[1:] - sp[:-1])
        assert torch.unique(slot * n + si.long()).numel() == si.numel()                    # no repeats in a row
        sp2, si2 = capi.csr_sampling(indptr, indices, seeds, k, False, seed=7777, stream_id=hop)
        assert torch.equal(sp, sp2) and torch.equal(si, si2)                               # cache is transparent
        u, (ls, ln) = capi.tensor_relabel([seeds, si])
        fsp, fsi, fu, fl = capi.sample_hop(indptr, indices, gp, gi, h, seeds, k, False, seed=7777, stream_id=hop)
        assert torch.equal(fsp, sp) and torch.equal(fsi, si) and torch.equal(fu, u) and torch.equal(fl, ln)
        assert torch.equal(u[: seeds.numel()], seeds) and torch.equal(u[ln], si.long())
        assert u.numel() == torch.unique(torch.cat([seeds, si.long()])).numel()
        seeds = u
    assert seeds.numel() > 100_000


@pytest.mark.parametrize("ptr", [np.int32, np.int64])
@pytest.mark.parametrize("rows,S,cached", [(40_000, 40_000, 0.0), (40_001, 9_000, 0.0), (3, 4_200, 0.0), (40_002, 40_000, 0.3),
                                           (40_003, 40_000, 0.97), (40_003, 40_000, 1.0), (120_000, 4_000, 0.0)])
def test_many_seeds_on_few_rows_of_host_memory(capi, ptr, rows, S, cached):
    """Row offsets that are copied to the GPU before the plan (many cold seeds), that are not because hardly a seed is
    cold, and that cannot pay (few seeds): all give what sampling the graph in device memory gives. The lengths
    end 0, 4, 8 and 12 bytes into a 16-byte word."""
    g = torch.Generator(device="cuda").manual_seed(rows + S)
    deg = torch.randint(0, 40, (rows,), device="cuda", generator=g)
    indptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(deg, 0, out=indptr[1:])
    indices = torch.randint(0, rows, (int(indptr[-1]),), device="cuda", generator=g)
    indptr = indptr.to(torch.int32 if ptr is np.int32 else torch.int64)
    seeds = torch.randint(0, rows, (S,), device="cuda", generator=g)
    want = capi.csr_sampling(indptr, indices, seeds, 5, False, seed=9)
    hp, hi = indptr.cpu().pin_memory(), indices.cpu().pin_memory()
    if cached == 0.0:
        got = capi.csr_sampling(hp, hi, seeds, 5, False, seed=9)
    else:
        for hot in (torch.randperm(rows, device="cuda", generator=g)[: int(rows * cached)],
                    torch.arange(int(rows * cached), device="cuda")):
            sub = capi.create_subcsr(hp, hi, hot)
            for layout in ("auto", "buckets"):
                h = capi.CUCOStaticHashmap(hot, torch.arange(hot.numel(), device="cuda"), 0.8, layout=layout)
                got = capi.csr_cache_sampling(hp, hi, sub[0], sub[1], h, seeds, 5, False, seed=9)
                assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    # offsets that start inside a 16-byte word are read where they are
    shifted = torch.empty(rows + 2, dtype=indptr.dtype, pin_memory=True)
    shifted[1:].copy_(indptr)
    got = capi.csr_sampling(shifted[1:], hi, seeds, 5, False, seed=9)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("order,copied", [("random", 1), ("sorted", 0), ("consecutive", 0), ("descending", 0), ("one row", 0)])
@pytest.mark.parametrize("mapped", [False, True])
def test_row_offsets_are_copied_only_for_the_lines_they_save(cabi, order, copied, mapped):
    """200,000 row offsets (1.6 MB) and 40,000 cold seeds: in random order each needs a line of its own (5 MB) and the
    offsets are copied first; seeds in id order share lines and are read where they are. Same samples either way."""
    import ctypes
    lib, stream = cabi.load(), cabi.current_stream()
    rows, S, k = 200_000, 40_000, 3
    g = torch.Generator(device="cuda").manual_seed(4)
    indptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.randint(0, 9, (rows,), device="cuda", generator=g), 0, out=indptr[1:])
    indices = torch.randint(0, rows, (int(indptr[-1]),), device="cuda", generator=g, dtype=torch.int32)
    seeds = {"random": torch.randperm(rows, device="cuda", generator=g)[:S],
             "sorted": torch.sort(torch.randperm(rows // 2, device="cuda", generator=g)[:S]).values,
             "consecutive": torch.arange(70_000, 70_000 + S, device="cuda"),
             "descending": torch.arange(S - 1, -1, -1, device="cuda"),
             "one row": torch.full((S,), 123, device="cuda")}[order].contiguous()
    handle, table = ctypes.c_void_p(), torch.empty(lib.shmt_hashmap_table_bytes(8, 0.5, 8, 8), dtype=torch.uint8, device="cuda")
    none = torch.arange(rows, rows + 8, device="cuda")     # (a map that holds none of the seeds)
    if mapped:
        cabi.check(lib.shmt_hashmap_create(ctypes.byref(handle), none.data_ptr(), none.data_ptr(), 8, 8, 8, 0.5, table.data_ptr(),
                                           table.numel(), stream))
    graph = (indptr.data_ptr(), 8, rows, indices.data_ptr(), 4) + ((indptr.data_ptr(), indices.data_ptr(), handle) if mapped
                                                                  else (None, None, None))
    plan = torch.empty(lib.shmt_sample_plan_bytes(S), dtype=torch.uint8, device="cuda")
    stage = torch.full((lib.shmt_sample_stage_bytes(rows, 8, S),), 255, dtype=torch.uint8, device="cuda")
    results = []
    for st in (stage, None):
        sp, si = torch.empty(S + 1, dtype=torch.int64, device="cuda"), torch.zeros(S * k, dtype=torch.int32, device="cuda")
        nnz = torch.zeros(1, dtype=torch.int64, pin_memory=True)
        cabi.check(lib.shmt_sample_staged(*graph, seeds.data_ptr(), 8, S, k, 0, 7, 0, sp.data_ptr(), si.data_ptr(), plan.data_ptr(),
                                          plan.numel(), st.data_ptr() if st is not None else None,
                                          st.numel() if st is not None else 0, nnz.data_ptr(), stream))
        torch.cuda.synchronize()
        results.append((sp, si, int(nnz)))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert results[0][2] == results[1][2]
    assert int(stage[:4].view(torch.int32)) == copied
    if copied:
        assert torch.equal(stage[128:128 + 8 * (rows + 1)].view(torch.int64), indptr)
    if mapped:
        lib.shmt_hashmap_destroy(handle)


def test_sub_graph_without_memory_for_row_starts(capi):
    """A sub-graph that fits is copied also where the 8 bytes per row that save host-link reads do not."""
    rows = 4_000_000
    indptr = torch.arange(0, 5 * rows + 1, 5, dtype=torch.int32)
    indices = torch.arange(5 * rows, dtype=torch.int32)
    seeds = torch.arange(rows, device="cuda")
    hp, hi = indptr.pin_memory(), indices.pin_memory()
    want = (5 * rows * 4 + (rows + 1) * 4) >> 20            # 80 MB + 16 MB
    total = torch.cuda.get_device_properties(0).total_memory
    for spare in (12, 40, 60):        # no room for the row starts (32 MB); for them alone; for all
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        try:
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + ((want + spare) << 20)) / total)
            gp, gi = capi.create_subcsr(hp, hi, seeds)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.equal(gp.cpu(), indptr) and torch.equal(gi.cpu(), indices)
        del gp, gi


@pytest.mark.parametrize("S,looked_at", [(5_000, False), (13_500, False), (13_600, True)])
def test_few_seeds_beside_a_map_are_not_looked_at(cabi, S, looked_at):
    """With a map the seeds are looked at only where a copy of the row offsets could save a good deal: 160,008 bytes
    of offsets and 1.5 MiB are 13,539 lines. (The flag in front of the staged offsets stays as it was otherwise.)"""
    import ctypes
    lib, stream = cabi.load(), cabi.current_stream()
    rows, k = 20_000, 3
    indptr = torch.arange(0, 2 * rows + 1, 2, device="cuda")
    indices = torch.arange(2 * rows, device="cuda", dtype=torch.int32)
    seeds = torch.randint(0, rows, (S,), device="cuda")
    handle, table = ctypes.c_void_p(), torch.empty(lib.shmt_hashmap_table_bytes(8, 0.5, 8, 8), dtype=torch.uint8, device="cuda")
    none = torch.arange(rows, rows + 8, device="cuda")
    cabi.check(lib.shmt_hashmap_create(ctypes.byref(handle), none.data_ptr(), none.data_ptr(), 8, 8, 8, 0.5, table.data_ptr(),
                                       table.numel(), stream))
    plan = torch.empty(lib.shmt_sample_plan_bytes(S), dtype=torch.uint8, device="cuda")
    stage = torch.full((max(128, lib.shmt_sample_stage_bytes(rows, 8, S)),), 255, dtype=torch.uint8, device="cuda")
    sp, si = torch.empty(S + 1, dtype=torch.int64, device="cuda"), torch.zeros(S * k, dtype=torch.int32, device="cuda")
    nnz = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    cabi.check(lib.shmt_sample_staged(indptr.data_ptr(), 8, rows, indices.data_ptr(), 4, indptr.data_ptr(), indices.data_ptr(),
                                      handle, seeds.data_ptr(), 8, S, k, 0, 7, 0, sp.data_ptr(), si.data_ptr(), plan.data_ptr(),
                                      plan.numel(), stage.data_ptr(), stage.numel(), nnz.data_ptr(), stream))
    torch.cuda.synchronize()
    assert int(nnz) == 2 * S and torch.equal(si[: 2 * S].view(S, 2).long(), torch.stack([2 * seeds, 2 * seeds + 1], 1))
    assert (int(stage[:4].view(torch.int32)) in (0, 1)) == looked_at
    lib.shmt_hashmap_destroy(handle)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("skew", [0, 3, 31])
@pytest.mark.parametrize("longest", [150, 700, 40_000])
def test_sub_graph_of_long_rows(capi, oracle, dtype, skew, longest):
    """Rows of several lines are copied line by line: rows that begin and end anywhere in a line, that fill lines exactly,
    empty ones, rows longer than a wave's chunk, and an index array that does not begin on a line."""
    g = np.random.default_rng(longest + skew)
    rows = 3000 if longest < 10_000 else 60
    deg = g.integers(longest // 2, longest + 1, rows)
    deg[g.integers(0, rows, rows // 10)] = 0
    deg[: 12] = [0, 1, 15, 16, 17, 31, 32, 33, 64, longest, 128, 0]
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    ids = torch.randint(0, 1 << 30, (int(indptr[-1]) + skew,), dtype=dtype).pin_memory()[skew:]
    hp = torch.from_numpy(indptr).pin_memory()
    for order in (np.arange(rows), g.permutation(rows)[: rows * 2 // 3], g.integers(0, rows, rows)):
        gp, gi = capi.create_subcsr(hp, ids, torch.from_numpy(order.astype(np.int64)).cuda())
        ep, ei = oracle.create_subcsr(indptr, ids.numpy(), order.astype(np.int64))
        assert np.array_equal(gp.cpu().numpy(), ep) and np.array_equal(gi.cpu().numpy(), ei)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_sub_graph_copy_stops_at_the_count_it_is_given(cabi, dtype):
    """A count below what the rows hold: that many elements are written and none behind them, also where the chunk in front of
    the last one ends within a few elements of the count (chunks start at multiples of 512 elements here)."""
    lib, size = cabi.load(), torch.empty(0, dtype=dtype).element_size()
    deg = torch.tensor([301, 0, 700, 333, 1500, 10])
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64), deg.cumsum(0)])
    indices = torch.randint(0, 1 << 30, (int(indptr[-1]) + 3,), dtype=dtype).cuda()[3:]     # (borders move off the multiples)
    rows, offsets, starts = torch.arange(6).cuda(), indptr.cuda(), indptr[:-1].contiguous().cuda()
    for nnz in (400, 1001, 1025, 1026, 1540, 1567, 2049, 2078, 2560, 2561, int(indptr[-1])):
        for begins in (None, starts.data_ptr()):
            out = torch.full((int(indptr[-1]) + 64,), -1, dtype=dtype, device="cuda")
            cabi.check(lib.shmt_subcsr_copy_rows(offsets.data_ptr(), indices.data_ptr(), 8, size, rows.data_ptr(), 8, 6,
                                                 offsets.data_ptr(), begins, nnz, out.data_ptr(), cabi.current_stream()))
            assert torch.equal(out[:nnz], indices[:nnz]) and bool((out[nnz:] == -1).all())


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("shape", ["empty runs", "hubs, then short rows", "hubs among short rows", "just few rows a chunk"])
def test_sub_graph_of_rows_of_any_lengths(capi, cabi, oracle, dtype, shape):
    """Long rows on average, but hubs beside rows of a few ids and runs of up to 9,000 empty rows (more rows than one look at 64
    of them, or at 64 * 64, covers): chunks that walk through their rows and chunks whose elements look for theirs, side by side."""
    g = np.random.default_rng(len(shape))
    hubs = lambda n: g.integers(3000, 9000, n)
    if shape == "empty runs":
        parts = [g.integers(0, 900, 40), np.zeros(9000), [1], np.zeros(62), [5], np.zeros(63), [700], np.zeros(64), hubs(180), np.zeros(4095),
                 [33], np.zeros(4097), hubs(20), np.zeros(300)]
    elif shape == "hubs, then short rows":
        parts = [hubs(200), g.integers(0, 8, 9000), hubs(1), g.integers(0, 3, 1000)]
    elif shape == "hubs among short rows":
        parts = [np.concatenate([hubs(1), g.integers(0, 9, int(g.integers(1, 90)))]) for _ in range(150)]
    else:   # (62 to 65 rows in a chunk of 512 to 4,096 elements, and the fewest bytes a row that are walked through)
        parts = [np.concatenate([np.full(int(g.integers(7, 66)), 64), hubs(1)]) for _ in range(60)]
    deg = np.concatenate(parts).astype(np.int64)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    assert indptr[-1] * 4 >= deg.size * 256
    ids = torch.randint(0, 1 << 30, (int(indptr[-1]) + 5,), dtype=dtype).pin_memory()[5:]
    hp = torch.from_numpy(indptr).pin_memory()
    for order in (np.arange(deg.size), g.permutation(deg.size)):
        at = torch.from_numpy(order).cuda()
        gp, gi = capi.create_subcsr(hp, ids, at)
        ep, ei = oracle.create_subcsr(indptr, ids.numpy(), order)
        assert np.array_equal(gp.cpu().numpy(), ep) and np.array_equal(gi.cpu().numpy(), ei)
        # (where nothing tells the rows' begins, they come from the row offsets)
        out, source, begins = torch.zeros_like(gi), ids.cuda(), hp.cuda()
        cabi.check(cabi.load().shmt_subcsr_copy(begins.data_ptr(), source.data_ptr(), 8, gi.element_size(), at.data_ptr(), 8, deg.size,
                                                gp.data_ptr(), gi.numel(), out.data_ptr(), cabi.current_stream()))
        assert torch.equal(out, gi)


def test_sub_graph_with_a_long_run_of_empty_rows_costs_what_its_ids_cost(capi):
    """200,000 empty rows in the middle of 13 M ids, and the same ids without them: a wave that stepped through them one by one
    took 20 times as long for the whole copy."""
    indices = torch.arange(13_000_000, dtype=torch.int32).pin_memory()

    def best_ms(empty):
        deg = torch.full((26_000,), 500)
        deg = torch.cat([deg[:13_000], torch.zeros(empty, dtype=torch.int64), deg[13_000:]])
        indptr = torch.cat([torch.zeros(1, dtype=torch.int64), deg.cumsum(0)])
        hp, rows = indptr.pin_memory(), torch.arange(deg.numel()).cuda()
        times = []
        for _ in range(5):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            gp, gi = capi.create_subcsr(hp, indices, rows)
            stop.record()
            stop.synchronize()
            times.append(start.elapsed_time(stop))
            assert torch.equal(gp.cpu(), indptr) and torch.equal(gi.cpu(), indices)
        return min(times)

    assert best_ms(200_000) < 4 * best_ms(0)
