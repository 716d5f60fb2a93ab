"""Relabel through hash partitions whose shares differ: ids are chosen by their hash so that a few partitions get nearly all of
them, or all, and many tiles have no id for a partition; bit-exact against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def tuning(cabi):
    lib = cabi.load()

    def set_(min_ids, slots_log2=0, rounds_log2=-1):
        cabi.check(lib.shmt_relabel_tuning(min_ids, slots_log2, rounds_log2))

    yield set_
    lib.shmt_relabel_tuning(0, 0, -1)


def _bin(ids):
    """Partition, among 256, of int64 ids (hash_id of the kernels)."""
    u = ids.astype(np.uint64)
    h = (u & np.uint64(0xFFFFFFFF)).astype(np.uint32) ^ ((u >> np.uint64(32)).astype(np.uint32) * np.uint32(0x9E3779B1))
    h ^= h >> np.uint32(16)
    h *= np.uint32(0x85EBCA6B)
    h ^= h >> np.uint32(13)
    h *= np.uint32(0xC2B2AE35)
    h ^= h >> np.uint32(16)
    return h >> np.uint32(24)


def _crowd(n, bins, share, dt, wide, rng):
    """n distinct-ish ids of which `share` lie in the first `bins` partitions."""
    pool = rng.integers(0, 2**31 - 1, size=n * 300 // max(bins, 1) + 4096).astype(np.int64)
    if wide:
        pool += rng.integers(0, 2, size=pool.size) << 40
    inside = pool[_bin(pool) < bins][:n]
    ids = np.where(rng.random(n) < share, inside[rng.integers(0, inside.size, size=n)], rng.choice(pool, size=n))
    return ids.astype(dt)


@pytest.mark.parametrize("n", [13_501, 60_000, 250_000])
@pytest.mark.parametrize("bins,share", [(1, 1.0), (1, 0.01), (3, 0.5), (100, 0.9)])
@pytest.mark.parametrize("dt,wide", [(np.int32, False), (np.int64, False), (np.int64, True)])
def test_crowded_partitions(capi, oracle, tuning, n, bins, share, dt, wide):
    rng = np.random.default_rng(n + bins)
    a = _crowd(n, bins, share, dt, wide, rng)
    tuning(8193)
    cut = n // 3
    u, labs = capi.tensor_relabel([torch.from_numpy(a[:cut].copy()).cuda(), torch.from_numpy(a[cut:].copy()).cuda()])
    eu, elabs = oracle.relabel([a[:cut], a[cut:]])
    assert np.array_equal(u.cpu().numpy(), eu)
    for l, e in zip(labs, elabs):
        assert np.array_equal(l.cpu().numpy(), e)


@pytest.mark.parametrize("slots_log2,rounds_log2", [(4, -1), (2, 0)])
@pytest.mark.parametrize("wide", [False, True])
def test_crowded_partition_that_does_not_fit_its_table(cabi, oracle, tuning, slots_log2, rounds_log2, wide):
    """Rounds and all pairs over the runs of many tiles, through the entry that takes one array."""
    lib, n = cabi.load(), 13_501
    ids = _crowd(n, 2, 0.3, np.int64, wide, np.random.default_rng(slots_log2))
    ids[::50] = -5
    tuning(8193, slots_log2, rounds_log2)
    total = torch.from_numpy(ids).cuda()
    sbytes = lib.shmt_relabel_scratch_bytes(n)
    scratch = torch.empty(sbytes, dtype=torch.uint8).cuda()
    unique, labels, count = torch.empty_like(total), torch.empty_like(total), torch.zeros(1, dtype=torch.int64).cuda()
    cabi.check(lib.shmt_relabel(total.data_ptr(), n, 8, scratch.data_ptr(), sbytes, unique.data_ptr(), labels.data_ptr(),
                                count.data_ptr(), cabi.current_stream()))
    eu, (el,) = oracle.relabel([ids])
    k = int(count.item())
    assert k == eu.size and np.array_equal(unique.cpu().numpy()[:k], eu) and np.array_equal(labels.cpu().numpy(), el)


@pytest.mark.parametrize("n_batches", [1, 5])
def test_crowded_partitions_in_hops(capi, oracle, tuning, n_batches):
    """Fused hops, alone and merged, on a graph whose neighbours all lie in two partitions: the same as by default, which goes
    by classes (the last hops are sized for 188,100 ids)."""
    rng = np.random.default_rng(3)
    n = 1 << 15
    nodes = np.arange(n, dtype=np.int64)
    few = nodes[_bin(nodes) < 2]
    deg = rng.integers(0, 40, size=n)
    indptr = torch.from_numpy(np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)).cuda()
    indices = torch.from_numpy(rng.choice(few, size=int(deg.sum())).astype(np.int32)).cuda()
    batches = [torch.from_numpy(rng.permutation(n)[:1900]).cuda() for _ in range(n_batches)]
    got = []
    for min_ids in (0, 8193):
        tuning(min_ids)
        got.append([capi.sample_hop(indptr, indices, None, None, None, batches[0], 10, False, seed=5),
                    *[hop for blocks in capi.sample_blocks(indptr, indices, None, None, None, batches, [10, 8], False,
                                                           seeds_rng=list(range(n_batches)), max_in_flight=8) for hop in blocks]])
        torch.cuda.synchronize()
    for x, y in zip(*got):
        assert len(x) == len(y)
        for p, q in zip(x, y):
            assert torch.equal(p, q)
