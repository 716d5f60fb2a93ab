"""Relabel of inputs between 8,192 and about a million ids, told apart by one class byte per id: against the oracle over
what decides the path inside (repeats that another element stands for, lists that overflow, tables that do not
hold their class), for ids that a separate launch classifies and for those that the pick kernel does."""
import numpy as np
import pytest
import torch

from test_gpu_relabel_partition import KINDS32, KINDS64, _ids, tuning  # noqa: F401

pytestmark = pytest.mark.gpu


def _check(capi, oracle, parts):
    u, labels = capi.tensor_relabel([torch.from_numpy(p).cuda() for p in parts])
    eu, elabels = oracle.relabel(parts)
    assert np.array_equal(u.cpu().numpy(), eu)
    for got, want in zip(labels, elabels):
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("n", [8193, 70_001, 524_288, 524_289, 1_000_000])
@pytest.mark.parametrize("dt,kind", [(np.int64, k) for k in KINDS64] + [(np.int32, k) for k in KINDS32])
def test_relabel_by_class_matches_oracle(capi, oracle, n, dt, kind):
    rng = np.random.default_rng(n)
    ids = _ids(kind, n, rng, dt)
    cut = int(rng.integers(1, n))
    _check(capi, oracle, [ids[:cut], ids[cut:]])


@pytest.mark.parametrize("distinct", [1, 100, 3000, 9000])
@pytest.mark.parametrize("n", [500_000, 900_000])
def test_more_elements_of_a_class_than_its_list_holds(capi, oracle, n, distinct):
    """A few ids, each in every tile: a class has up to a hundred times the elements that its share of distinct ids suggests."""
    _check(capi, oracle, [np.random.default_rng(distinct).integers(0, distinct, n).astype(np.int64) * 7919])


def test_ids_that_come_in_every_tile_are_no_slower(cabi):
    """A thousand ids put up to 5,000 elements into a class, ten thousand about 2,000: the list has room for either. (Where the
    elements beyond 4,096 went into the table one by one: 61 us against 37.)"""
    lib, n = cabi.load(), 520_000
    g = torch.Generator(device="cuda").manual_seed(1)
    sbytes = lib.shmt_relabel_scratch_bytes(n)
    scratch = torch.empty(sbytes, dtype=torch.uint8, device="cuda")
    unique, labels = (torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(2))
    count = torch.zeros(1, dtype=torch.int64, device="cuda")
    took = []
    for distinct in (1_000, 10_000):
        ids = (torch.randint(0, distinct, (n,), device="cuda", generator=g) * 7919).to(torch.int32)
        runs = []
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(20):
                cabi.check(lib.shmt_relabel(ids.data_ptr(), n, 4, scratch.data_ptr(), sbytes, unique.data_ptr(), labels.data_ptr(),
                                            count.data_ptr(), cabi.current_stream()))
            b.record()
            torch.cuda.synchronize()
            runs.append(a.elapsed_time(b))
        assert int(count.item()) == distinct
        took.append(min(runs))
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


@pytest.mark.parametrize("dt,kind", [(np.int32, "hub"), (np.int64, "spread32"), (np.int64, "wide")])
def test_inputs_that_keep_the_table_in_memory(capi, oracle, dt, kind):
    _check(capi, oracle, [_ids(kind, 7_400_000, np.random.default_rng(7), dt)])
