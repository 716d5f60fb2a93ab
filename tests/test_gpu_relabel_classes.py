"""Relabel of 8,193 to 393,216 ids (for a hop up to 524,287, sized by a loose bound up to 2,097,152), told apart by one class byte per id:
against the oracle over what decides the path inside (repeats that another element stands for, lists that overflow, tables
that do not hold their class), for ids that a separate launch classifies and for those that the pick kernel does."""
import numpy as np
import pytest
import torch

from test_gpu_relabel_crowded import _bin
from test_gpu_relabel_partition import KINDS32, KINDS64, _ids, tuning  # noqa: F401

pytestmark = pytest.mark.gpu


def _check(capi, oracle, parts):
    u, labels = capi.tensor_relabel([torch.from_numpy(p).cuda() for p in parts])
    eu, elabels = oracle.relabel(parts)
    assert np.array_equal(u.cpu().numpy(), eu)
    for got, want in zip(labels, elabels):
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("n", [8193, 70_001, 393_216, 393_217])      # (the last one: the first that takes partitions)
@pytest.mark.parametrize("dt,kind", [(np.int64, k) for k in KINDS64] + [(np.int32, k) for k in KINDS32])
def test_relabel_by_class_matches_oracle(capi, oracle, n, dt, kind):
    rng = np.random.default_rng(n)
    ids = _ids(kind, n, rng, dt)
    cut = int(rng.integers(1, n))
    _check(capi, oracle, [ids[:cut], ids[cut:]])


@pytest.mark.parametrize("distinct", [1, 100, 3000, 9000])
@pytest.mark.parametrize("n", [200_000, 393_216])
def test_more_elements_of_a_class_than_its_list_holds(capi, oracle, n, distinct):
    """A few ids, each in every tile: a class has up to a hundred times the elements that its share of distinct ids suggests."""
    _check(capi, oracle, [np.random.default_rng(distinct).integers(0, distinct, n).astype(np.int64) * 7919])


def test_few_neighbours_are_hardly_slower_than_many(capi, oracle):
    """A hundred ids that come in every wave of the pick kernel put up to 8,000 elements into a class, ten thousand about
    2,000: the list has room for either. (Where those beyond 4,096 went into the table one by one: 98 us against 65.)"""
    n, n_seeds = 200_000, 19_000
    g = torch.Generator(device="cuda").manual_seed(1)
    indptr = torch.arange(0, 30 * n + 1, 30, device="cuda")
    seeds = torch.randperm(n, device="cuda", generator=g)[:n_seeds].to(torch.int32)
    took = []
    for distinct in (100, 10_000):
        indices = torch.randint(0, distinct, (30 * n,), device="cuda", generator=g).to(torch.int32)
        runs = []
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(20):
                hop = capi.sample_hop(indptr, indices, None, None, None, seeds, 25, False, seed=11)
            b.record()
            torch.cuda.synchronize()
            runs.append(a.elapsed_time(b))
        took.append(min(runs))
        eu, (_, el) = oracle.relabel([seeds.cpu().numpy(), hop[1].cpu().numpy()])
        assert np.array_equal(hop[2].cpu().numpy(), eu) and np.array_equal(hop[3].cpu().numpy(), el)
    assert took[0] < 1.3 * took[1]


@pytest.mark.parametrize("slots_log2,rounds_log2", [(6, -1), (3, -1), (4, 2), (2, 0)])
@pytest.mark.parametrize("kind", ["spread32", "wide", "minus_one", "hub"])
def test_class_that_does_not_fit_its_table(capi, oracle, tuning, slots_log2, rounds_log2, kind):  # noqa: F811
    tuning(1 << 40, slots_log2, rounds_log2)
    _check(capi, oracle, [_ids(kind, 40_000, np.random.default_rng(slots_log2), np.int64)])


@pytest.mark.parametrize("idx_dt,kind", [(np.int32, "spread32"), (np.int32, "negative"), (np.int32, "hub"), (np.int64, "spread32"),
                                         (np.int64, "wide"), (np.int64, "hub"), (np.int64, "minus_one"), (np.int64, "uint32_max")])
@pytest.mark.parametrize("seed_dt", [torch.int32, torch.int64])
@pytest.mark.parametrize("k", [5, 25, 40, 70])
def test_hop_classifies_what_it_picks(capi, oracle, idx_dt, kind, seed_dt, k):
    """k = 70: one wave per seed, which leaves the classes to a launch of their own."""
    rng = np.random.default_rng(k)
    deg = rng.integers(0, 3 * k, 4000)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    indices = _ids(kind, int(indptr[-1]), rng, idx_dt)
    t = lambda a: torch.from_numpy(a).cuda()
    seeds = torch.randint(0, 4000, (3000,), device="cuda").to(seed_dt)
    sp, si, unique, labels = capi.sample_hop(t(indptr), t(indices), None, None, None, seeds, k, False, seed=11)[:4]
    esp, esi = capi.csr_sampling(t(indptr), t(indices), seeds, k, False, seed=11)
    assert torch.equal(sp, esp) and torch.equal(si, esi)
    wide = np.int64 if seed_dt == torch.int64 or idx_dt == np.int64 else np.int32
    eu, (_, el) = oracle.relabel([seeds.cpu().numpy().astype(wide), esi.cpu().numpy().astype(wide)])
    assert np.array_equal(unique.cpu().numpy(), eu) and np.array_equal(labels.cpu().numpy(), el)


@pytest.mark.parametrize("dt", [torch.int32, torch.int64])
@pytest.mark.parametrize("n_seeds,n_batches,empty,slots_log2,rounds_log2", [
    (1000, 1, 0.0, 0, -1), (3300, 1, 0.0, 0, -1), (3300, 3, 0.0, 0, -1), (1000, 2, 0.0, 8, -1), (3300, 1, 0.0, 10, 1),
    (1000, 3, 0.95, 2, 0)])
def test_hops_of_a_loose_bound(capi, oracle, tuning, dt, n_seeds, n_batches, empty, slots_log2, rounds_log2):  # noqa: F811
    """Second hops sized for 600,000 or 1,980,000 ids, alone and two or three to a launch: the larger table. Nearly all
    neighbours are of one class, with more elements than its list holds, and more ids than a lowered table; where most
    rows are empty, few enough for a table of four slots to end in comparing all pairs."""
    tuning(1 << 40, slots_log2, rounds_log2)
    n, picks = 600_000, [24, 23]
    g = torch.Generator(device="cuda").manual_seed(n_seeds + n_batches)
    nodes = np.arange(n)
    few = torch.from_numpy(nodes[_bin(nodes) == 0]).cuda()     # (the first 256th of the hashes: within the first class of 255)
    deg = torch.randint(20, 40, (n,), device="cuda", generator=g) * (torch.rand(n, device="cuda", generator=g) >= empty)
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), deg.cumsum(0)])
    nnz = int(indptr[-1])
    at = torch.randint(0, few.numel(), (nnz,), device="cuda", generator=g)
    other = torch.randint(0, n, (nnz,), device="cuda", generator=g)
    indices = torch.where(torch.rand(nnz, device="cuda", generator=g) < 0.95, few[at], other).to(dt)
    batches = [torch.randperm(n, device="cuda", generator=g)[:n_seeds].to(dt) for _ in range(n_batches)]
    got = capi.sample_blocks(indptr, indices, None, None, None, batches, picks, False, seeds_rng=list(range(n_batches)),
                             max_in_flight=8)
    np_dt = np.int32 if dt == torch.int32 else np.int64
    for seeds, hops in zip(batches, got):
        frontier = seeds.cpu().numpy()
        for _, picked, unique, labels in (hop[:4] for hop in hops):
            picked = picked.cpu().numpy().astype(np_dt)
            eu, (_, el) = oracle.relabel([frontier, picked])
            assert np.array_equal(unique.cpu().numpy(), eu) and np.array_equal(labels.cpu().numpy(), el)
            frontier = eu
        in_class = int((_bin(picked.astype(np.int64)) == 0).sum())
        assert (in_class > 50_000) if empty == 0.0 else (in_class < 20_000)


@pytest.mark.parametrize("dt,kind", [(np.int32, "hub"), (np.int64, "spread32"), (np.int64, "wide")])
def test_inputs_that_keep_the_table_in_memory(capi, oracle, dt, kind):
    _check(capi, oracle, [_ids(kind, 7_400_000, np.random.default_rng(7), dt)])
