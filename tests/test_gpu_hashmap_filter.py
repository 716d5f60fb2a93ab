"""Bulk lookups in tables with a presence filter (narrow tables built by partitions, from 2^20 pairs on), asked by calls of 2^21
requests and more: at every share of absent requests, with which the filter is used or not, they answer as the pairs say."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _keys(n, bits, g):
    pool = torch.unique(torch.randint(0, 1 << bits, (n + n // 4 + 64,), device="cuda", generator=g))
    return pool[torch.randperm(pool.numel(), device="cuda", generator=g)].contiguous()


def _check(h, keys, others, nq, share, g, out_dtype=torch.int64):
    """Requests of which `share` are keys, in runs of 5,000 of one kind and mixed ones in turn."""
    at = torch.randint(0, keys.numel(), (nq,), device="cuda", generator=g)
    member = torch.rand(nq, device="cuda", generator=g) < share
    runs = (torch.arange(nq, device="cuda") // 5000) % 3
    member = torch.where(runs == 0, member, runs == 1)
    other = others[torch.randint(0, others.numel(), (nq,), device="cuda", generator=g)]
    got = h.query(torch.where(member, keys[at], other))
    assert got.dtype == out_dtype and torch.equal(got.to(torch.int64), torch.where(member, at, -1))


# pairs, bits of a key, load: just no filter and just one; words of two buckets; packed and 32-bit words
@pytest.mark.parametrize("n,bits,load", [((1 << 20) - 1, 40, 0.5), (1 << 20, 40, 0.5), ((1 << 20) + 77, 31, 0.5),
                                         ((1 << 21) + 13, 45, 0.3), (6_000_000, 42, 0.8)])
@pytest.mark.parametrize("share", [0.0, 0.6, 1.0])
def test_lookups_with_absent_requests(capi, n, bits, load, share):
    g = torch.Generator(device="cuda").manual_seed(n)
    pool = _keys(n + 100_000, bits, g)
    keys, others = pool[:n].contiguous(), torch.cat([pool[n:], torch.tensor([-1, 1 << 62, -2**63], device="cuda")])
    h = capi.CUCOStaticHashmap(keys, torch.arange(n, device="cuda"), load)
    assert h.layout() == "buckets"
    for nq in ((1 << 21) - 1, 1 << 21, 3_000_001, 4_000_000):      # (the first one does not ask the filter)
        _check(h, keys, others, nq, share, g)


def test_no_share_of_keys_makes_lookups_slower_than_keys_alone(capi):
    """A filter that only some of the waves ask loses its place in the caches: 65 per cent of keys took 10 per cent longer than
    keys alone, where it is either of use or left alone."""
    g = torch.Generator(device="cuda").manual_seed(9)
    n, nq = 1 << 22, 1 << 24
    pool = _keys(n + 500_000, 40, g)
    keys, others = pool[:n].contiguous(), pool[n:]
    h = capi.CUCOStaticHashmap(keys, torch.arange(n, device="cuda"), 0.5)

    def best_ms(share):
        member = torch.rand(nq, device="cuda", generator=g) < share
        q = torch.where(member, keys[torch.randint(0, n, (nq,), device="cuda", generator=g)],
                        others[torch.randint(0, others.numel(), (nq,), device="cuda", generator=g)])
        times = []
        for _ in range(12):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            h.query(q)
            stop.record()
            stop.synchronize()
            times.append(start.elapsed_time(stop))
        return min(times)

    alone = best_ms(1.0)
    for share in (0.5, 0.6, 0.65, 0.7, 0.8):
        assert best_ms(share) < 1.05 * alone, share


@pytest.mark.parametrize("n,filtered", [((1 << 20) - 1, False), (1 << 20, True)])
def test_smallest_table_with_a_filter(cabi, n, filtered):
    lib = cabi.load()
    keys = _keys(n, 40, torch.Generator(device="cuda").manual_seed(n))[:n].contiguous()
    vals = torch.arange(n, device="cuda")
    sb = lib.shmt_hashmap_plan_scratch_bytes(n)
    scratch, lay = torch.empty(sb, dtype=torch.uint8, device="cuda"), cabi.HashmapLayout()
    cabi.check(lib.shmt_hashmap_plan(keys.data_ptr(), vals.data_ptr(), n, 8, 8, 0.5, scratch.data_ptr(), sb, ctypes.byref(lay),
                                     cabi.current_stream()))
    assert (lay.kind, lay.slot_bytes) == (0, 8)
    assert lay.table_bytes - lib.shmt_hashmap_table_bytes(n, 0.5, 4, 4) == (n // 8 * 4 if filtered else 0)


def test_int32_pairs(capi):
    g = torch.Generator(device="cuda").manual_seed(5)
    n = 1_300_000
    pool = _keys(n + 50_000, 31, g).to(torch.int32)
    keys, others = pool[:n].contiguous(), pool[n:]
    h = capi.CUCOStaticHashmap(keys, torch.arange(n, device="cuda", dtype=torch.int32), 0.5)
    _check(h, keys, others, 3_000_000, 0.3, g, torch.int32)


def test_repeated_keys_without_room(capi):
    """Pairs that find no room in their partition's reserve are filtered in too."""
    g = torch.Generator(device="cuda").manual_seed(6)
    n = 1 << 20
    pool = _keys(n, 40, g)
    keys = torch.cat([pool[: n // 2], pool[:17].repeat(n // 34 + 1)[: n // 2]])[torch.randperm(n, device="cuda", generator=g)]
    h = capi.CUCOStaticHashmap(keys.contiguous(), torch.arange(n, device="cuda"), 0.5)
    q = torch.cat([keys, pool[n // 2:n], keys, pool[n // 2:n]])[torch.randperm(3 * n, device="cuda", generator=g)].contiguous()
    got = h.query(q)
    assert torch.equal(got >= 0, torch.isin(q, keys)) and torch.equal(keys[got[got >= 0]], q[got >= 0])


def test_table_memory_decides_on_the_filter(cabi):
    """With the memory that the plan names there is a filter, with that of the buckets alone there is none; either way, and
    built without scratch memory, lookups are the same and nothing behind the given memory is written."""
    lib, stream = cabi.load(), cabi.current_stream()
    g = torch.Generator(device="cuda").manual_seed(7)
    n = (1 << 20) + 5
    pool = _keys(n + 10_000, 40, g)
    keys, vals = pool[:n].contiguous(), torch.arange(n, device="cuda")
    sb = lib.shmt_hashmap_plan_scratch_bytes(n)
    scratch = torch.empty(sb, dtype=torch.uint8, device="cuda")
    lay = cabi.HashmapLayout()
    cabi.check(lib.shmt_hashmap_plan(keys.data_ptr(), vals.data_ptr(), n, 8, 8, 0.5, scratch.data_ptr(), sb, ctypes.byref(lay), stream))
    buckets = lib.shmt_hashmap_table_bytes(n, 0.5, 4, 4)          # (8-byte slots as well)
    planned = lay.table_bytes
    assert (lay.kind, lay.slot_bytes) == (0, 8) and buckets < planned <= buckets + buckets // 32 + 128
    need = lib.shmt_hashmap_build_scratch_bytes(ctypes.byref(lay), n, 0.5)
    build = torch.empty(need, dtype=torch.uint8, device="cuda")
    at = torch.randint(0, n, (2_500_000,), device="cuda", generator=g)
    q = torch.where(at % 2 == 0, keys[at], pool[n + at % 10_000]).contiguous()
    want = torch.where(at % 2 == 0, at, -1)
    for said, given, with_scratch, used in ((planned, planned, True, planned), (planned, buckets, True, buckets),
                                            (buckets, planned, True, buckets), (planned, planned, False, buckets)):
        lay.table_bytes = said
        memory = torch.full((planned + 128,), 0x5A, dtype=torch.uint8, device="cuda")
        handle = ctypes.c_void_p()
        cabi.check(lib.shmt_hashmap_create_planned_scratch(
            ctypes.byref(handle), ctypes.byref(lay), keys.data_ptr(), vals.data_ptr(), n, 8, 8, 0.5, memory.data_ptr(), given,
            build.data_ptr() if with_scratch else None, need if with_scratch else 0, stream))
        out = torch.empty_like(q)
        cabi.check(lib.shmt_hashmap_query(handle, q.data_ptr(), 8, q.numel(), out.data_ptr(), stream))
        assert torch.equal(out, want) and lib.shmt_hashmap_used_bytes(handle) == buckets
        assert bool((memory[used:] == 0x5A).all())
        lib.shmt_hashmap_destroy(handle)


def test_map_whose_buckets_alone_fit(capi):
    """Where there is memory for the buckets (64 MiB) but none for the filter behind them, the map is built without one."""
    g = torch.Generator(device="cuda").manual_seed(8)
    n = 1 << 22
    pool = _keys(n + 100_000, 40, g)
    keys, vals = pool[:n].contiguous(), torch.arange(n, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    before = torch.cuda.memory_allocated()
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (65 << 20)) / total)
        h = capi.CUCOStaticHashmap(keys, vals, 0.5)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.cuda.memory_allocated() - before == 64 << 20      # (no filter)
    filtered = capi.CUCOStaticHashmap(keys, vals, 0.5)
    assert torch.cuda.memory_allocated() - before == (64 + 66) << 20
    for each in (h, filtered):
        assert each.memory_usage() == 64 << 20
        _check(each, keys, pool[n:], 2_500_000, 0.5, g)
