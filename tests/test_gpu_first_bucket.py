"""Finds that rely on the table's first-bucket rule (2^22 lookups or more on a table that nothing was
erased from, resized or loaded since it was empty) against the same lookups in smaller calls, which
read in the reference order: values and flags bit for bit, also for copies of one key in both its
buckets, under each rule and under none, and where an erase on another stream, a captured find or
a refill could leave the rule behind. Each large find is checked to have taken the rule that the
table keeps then (NONE where it keeps none, or is too small to gain)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LARGE = 1 << 22
NONE, START, FILL = 0, 1, 2


@pytest.fixture(scope="module")
def D():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import databases_gpu_amd as D

    D.load()
    return D


def keys(lo, hi, seed=3):
    from databases_gpu_amd.workload import keys_range

    return keys_range(lo, hi, seed, torch.device("cuda", 0))


def lookups(n, stored, seed=0):
    """n lookups of keys(0, 2 * stored): about half of them stored."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    pool = torch.cat([keys(0, 2 * stored), torch.tensor([0, -1], dtype=torch.int32, device="cuda")])
    return pool[torch.randint(0, pool.numel(), (n,), generator=g, device="cuda")]


def last_rule(t):
    """The rule of the last find of a table, a group or a plan's graph."""
    kind = {"DyCuckoo": "", "DyCuckooWide": "wide_", "DyCuckooGroup": "group_", "DyCuckooWideGroup": "wide_group_",
            "GroupPlan": "plan_"}[type(t).__name__]
    f = getattr((t.group if kind == "plan_" else t).lib, f"dyc_internal_{kind}rule")
    f.restype, f.argtypes = ctypes.c_uint32, [ctypes.c_void_p]
    return f(t.h)


def both_ways(t, q, rule):
    """The large find, which takes `rule`, checked against small ones."""
    v, h = t.find(q)
    assert last_rule(t) == rule
    sv, sh = zip(*(t.find(x) for x in torch.split(q, LARGE - 1)))
    assert last_rule(t) == NONE
    assert torch.equal(h, torch.cat(sh)) and torch.equal(v, torch.cat(sv))
    return v, h


@pytest.mark.parametrize("d", [2, 4, 6])
@pytest.mark.parametrize("order", [0, 3])
def test_same_as_the_reference_order(D, order, d):
    print(f"\n[gpu-case] first-bucket rule d={d} insert_order={order}", flush=True)
    m = 1 << 21
    t = D.DyCuckoo(int(m / (0.6 if d == 2 else 0.65)), subtables=d, insert_order=order, kick_bound=0, auto_resize=0)
    # 32-bit keys all start in one of two subtables, so no find relies on that
    start = NONE if d == 2 else START
    kept = FILL if order == 3 else start
    k = keys(0, m)
    q = lookups(LARGE + 77, m, d)
    _, h = both_ways(t, q, FILL)  # empty
    assert not h.any()
    t.insert(k, k ^ 1)
    _, h = both_ways(t, q, kept)
    # a second copy of some keys (enough of them for a bulk fill): where the first bucket is full, in the
    # other one
    t.insert(k[: m // 4], k[: m // 4] ^ 2)
    both_ways(t, q, kept)
    # entries under the other rule (too few for a bulk fill)
    t.configure(insert_order=3 - order)
    extra = keys(3 * m, 3 * m + m // 32)
    t.insert(extra, extra)
    both_ways(t, torch.cat([q, extra]), NONE if order == 3 else start)
    # erased slots: the rule is gone
    gone = t.erase(k[: m // 2])
    assert gone.all()
    _, h2 = both_ways(t, q, NONE)
    assert int(h2.sum()) < int(h.sum())
    t.insert(k[: m // 2], k[: m // 2] ^ 3)
    both_ways(t, q, NONE)
    # emptied and filled again: the rule is back
    t.clear()
    t.insert(k, k ^ 4)
    v, h = both_ways(t, q, start if order == 3 else FILL)
    t.resize_up()
    v2, h2 = both_ways(t, q, NONE)
    assert torch.equal(h, h2) and torch.equal(v, v2)
    assert t.resize_down()
    both_ways(t, q, NONE)
    t.load(t.dump())
    both_ways(t, q, NONE)
    t.close()


def probes(t, q):
    """Buckets the last find's order reads for q."""
    f = t.lib.dyc_internal_wide_probes if q.dtype == torch.int64 else t.lib.dyc_internal_probes
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64,
                                           ctypes.POINTER(ctypes.c_uint64), ctypes.c_void_p]
    out = ctypes.c_uint64()
    torch.cuda.synchronize()
    assert f(t.h, q.data_ptr(), q.numel(), ctypes.byref(out), None) == 0
    return out.value


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("order", [0, 3])
def test_buckets_counted_are_those_the_find_reads(D, order, bits):
    print(f"\n[gpu-case] buckets a find reads, {bits}-bit keys, insert_order={order}", flush=True)
    from databases_gpu_amd.workload import u32_to_i64

    m = 1 << 21
    t = (D.DyCuckoo if bits == 32 else D.DyCuckooWide)(int(m / 0.8), insert_order=order, kick_bound=0, auto_resize=0)
    k, q = keys(0, m), lookups(LARGE, m)
    valid = int(((q != 0) & (q != -1)).sum())
    if bits == 64:
        k, q = u32_to_i64(k), u32_to_i64(q)  # 0xffffffff is no reserved 64-bit key
        valid = int((q != 0).sum())
    t.find(q)
    assert last_rule(t) == FILL and probes(t, q) == valid  # empty: every first bucket ends the search
    t.insert(k, k)
    t.find(q[:5])
    reference = probes(t, q)
    t.find(q)
    assert last_rule(t) == (FILL if order == 3 else START)
    assert valid < probes(t, q) < reference < 2 * valid
    if bits == 32:
        assert reference == t.probe_count(q)[0]
    t.close()


@pytest.mark.parametrize("bits", [32, 64])
def test_small_tables_read_in_the_reference_order(D, bits):
    print(f"\n[gpu-case] first-bucket rule, small table of {bits}-bit keys", flush=True)
    from databases_gpu_amd.workload import u32_to_i64

    m = 1 << 18
    t = (D.DyCuckoo if bits == 32 else D.DyCuckooWide)(int(m / 0.8), insert_order=3, kick_bound=0, auto_resize=0)
    k, q = keys(0, m), lookups(LARGE, m)
    if bits == 64:
        k, q = u32_to_i64(k), u32_to_i64(q)
    t.insert(k, k)
    both_ways(t, q, NONE)
    t.close()


@pytest.mark.parametrize("d", [2, 4])
@pytest.mark.parametrize("order", [0, 3])
def test_wide_tables(D, order, d):
    print(f"\n[gpu-case] first-bucket rule, wide d={d} insert_order={order}", flush=True)
    m = 1 << 20
    t = D.DyCuckooWide(int(m / (0.6 if d == 2 else 0.65)), subtables=d, insert_order=order, kick_bound=0, auto_resize=0)
    wide = lambda x: x.long() * 0x1_0000_0001 ^ 0x55  # noqa: E731
    kept = FILL if order == 3 else START
    k = wide(keys(0, m))
    q = torch.cat([wide(lookups(LARGE + 5, m, d)), torch.tensor([0, -1], device="cuda")])
    _, h = both_ways(t, q, FILL)
    assert not h.any()
    t.insert(k, k ^ 1)
    both_ways(t, q, kept)
    t.insert(k[: m // 4], k[: m // 4] ^ 2)
    both_ways(t, q, kept)
    t.upsert(k[: m // 16], k[: m // 16] ^ 3)  # under the start rule
    both_ways(t, q, NONE if order == 3 else START)
    assert t.erase(k[: m // 2]).all()
    both_ways(t, q, NONE)
    t.clear()
    t.insert(k, k ^ 4)
    v, h = both_ways(t, q, kept)
    t.resize_up()
    v2, h2 = both_ways(t, q, NONE)
    assert torch.equal(h, h2) and torch.equal(v, v2)
    t.close()


def test_upsert_and_host_inserts_keep_the_start_rule(D):
    print("\n[gpu-case] first-bucket rule, upsert and host inserts", flush=True)
    m = 1 << 21
    t = D.DyCuckoo(int(m / 0.8), insert_order=0, kick_bound=15, auto_resize=0)
    k = keys(0, m)
    q = lookups(LARGE, m)
    t.upsert(k[: m // 4], k[: m // 4])
    t.insert_host(k[m // 4: m // 2].cpu().numpy(), k[m // 4: m // 2].cpu().numpy())
    t.insert_async(k[m // 2:], k[m // 2:])
    t.upsert(k[: m // 4], k[: m // 4] ^ 9)
    both_ways(t, q, START)
    t.close()


def test_erase_on_another_stream_waits_for_the_find(D):
    """Keys that are not erased are found by a large find that an erase on another stream follows at
    once, although the erase frees slots in their first buckets."""
    print("\n[gpu-case] first-bucket rule, erase on another stream", flush=True)
    m = 1 << 21
    k = keys(0, m)
    stay, go = k[: m // 2], k[m // 2:]
    reps = 16
    q = stay.repeat(reps)  # 2^24 lookups
    t = D.DyCuckoo(int(m / 0.9), insert_order=3, kick_bound=0, auto_resize=0)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        t.clear()
        t.insert(k, k ^ 5)
        torch.cuda.synchronize()
        v, h = t.find(q, stream=a)
        assert last_rule(t) == FILL
        gone = t.erase(go, stream=b)
        torch.cuda.synchronize()
        assert gone.all() and h.all() and torch.equal(v, q ^ 5)
        v, h = both_ways(t, k.repeat(4), NONE)
        assert torch.equal(h.view(4, m)[0].bool(), torch.arange(m, device="cuda") < m // 2)
    t.close()


def test_captured_find_is_replayed_after_an_erase(D):
    print("\n[gpu-case] first-bucket rule, captured find", flush=True)
    m = 1 << 21
    k = keys(0, m)
    q = lookups(LARGE, m)
    t = D.DyCuckoo(int(m / 0.9), insert_order=3, kick_bound=0, auto_resize=0)
    t.insert(k, k)
    v = torch.empty_like(q)
    h = torch.empty(q.numel(), dtype=torch.uint8, device="cuda")
    t.find(q, v, h)
    assert last_rule(t) == FILL
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        t.find(q, v, h)
        assert last_rule(t) == NONE
    for part in torch.split(k, m // 3):
        t.erase(part)
        g.replay()
        torch.cuda.synchronize()
        sv, sh = zip(*(t.find(x) for x in torch.split(q, LARGE // 2)))
        assert torch.equal(h, torch.cat(sh)) and torch.equal(v, torch.cat(sv))
    t.close()


@pytest.mark.parametrize("order", [0, 3])
@pytest.mark.parametrize("bits", [32, 64])
def test_groups(D, bits, order):
    from databases_gpu_amd.table import DyCuckooGroup, DyCuckooWideGroup

    print(f"\n[gpu-case] first-bucket rule, groups bits={bits} insert_order={order}", flush=True)
    # one lookup for three keys: the tables in flight on an XCD are more than its L2 holds, so the group's
    # finds rely on the rule
    sizes = np.random.default_rng(1).integers(0, 1_300_000, size=24)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(off[-1])
    k = keys(0, n)
    pick = torch.cat([torch.arange(int(off[i]), int(off[i + 1]), 3, device="cuda") for i in range(sizes.size)])
    fsizes = -(-sizes // 3)
    foff = np.concatenate([[0], np.cumsum(fsizes)]).astype(np.uint64)
    assert LARGE < pick.numel() == int(foff[-1]) < 1 << 24
    q = torch.where(torch.rand(pick.numel(), device="cuda") < 0.5, keys(n, n + pick.numel()), k[pick])
    if bits == 64:
        k, q = k.long() * 0x9E3779B1 | 1, q.long() * 0x9E3779B1 | 1
    g = (DyCuckooGroup if bits == 32 else DyCuckooWideGroup)((sizes / 0.85).astype(np.uint64) + 128,
                                                             insert_order=order, kick_bound=0)

    def parts():
        out = []
        for lo in range(0, sizes.size, 4):
            some = np.where((np.arange(sizes.size) >= lo) & (np.arange(sizes.size) < lo + 4), fsizes, 0)
            a, b = int(foff[lo]), int(foff[min(lo + 4, sizes.size)])
            assert b - a < LARGE
            out.append(g.find(q[a:b].contiguous(), np.concatenate([[0], np.cumsum(some)]).astype(np.uint64)))
            assert last_rule(g) == NONE
        return torch.cat([x[0] for x in out]), torch.cat([x[1] for x in out])

    for step in range(3):
        if step == 2:
            g.clear()
        if step != 1:
            g.insert(k, k ^ step, off)
        else:
            erased = torch.arange(n, device="cuda") % 3 == 0
            g.erase(torch.where(erased, k, torch.zeros_like(k)), off)
        v, h = g.find(q, foff)
        assert last_rule(g) == (NONE if step == 1 else FILL if order == 3 else START)
        sv, sh = parts()
        assert torch.equal(h, sh) and torch.equal(v, sv)
    g.close()


def test_plan_relies_on_its_own_fill(D):
    from databases_gpu_amd.table import DyCuckooGroup

    print("\n[gpu-case] first-bucket rule, plans", flush=True)
    for order in (0, 3):
        sizes = np.random.default_rng(2).integers(100_000, 300_000, size=9)
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
        n = int(off[-1])
        k = keys(0, n)
        # as many lookups as keys, which find the tables in L2, and few of them
        for every, rule in ((1, NONE), (16, FILL if order == 3 else START)):
            pick = torch.cat([torch.arange(int(off[i]), int(off[i + 1]), every, device="cuda") for i in range(9)])
            foff = np.concatenate([[0], np.cumsum(-(-sizes // every))]).astype(np.uint64)
            miss = torch.rand(pick.numel(), device="cuda") < 0.4
            q = torch.where(miss, keys(n, n + pick.numel()), k[pick])
            g = DyCuckooGroup((sizes / 0.85).astype(np.uint64) + 128, insert_order=order, kick_bound=0)
            p = g.plan(k, k ^ 7, off, q, foff)
            assert last_rule(p) == rule
            for _ in range(3):
                p.run()
                assert torch.equal(p.out_hit.bool(), ~miss)
                assert torch.equal(p.out_vals, torch.where(miss, torch.zeros_like(q), q ^ 7))
                g.erase(k, off)  # eager work between the replays
            g.close()


@pytest.mark.parametrize("d", [3, 4])
@pytest.mark.parametrize("kick_bound", [0, 15])
def test_small_tables_looked_up_in_large_calls(D, kick_bound, d):
    """Tables of at most 1024 buckets, whose inserts spread a wave's lanes over a bucket's empty slots:
    each stored key is found by a find that stops at a first bucket with a free slot. The large
    tables bring the group's mean to where its finds rely on the rule."""
    from databases_gpu_amd.table import DyCuckooGroup

    print(f"\n[gpu-case] first-bucket rule, small tables d={d} kick_bound={kick_bound}", flush=True)
    sizes = np.concatenate([np.random.default_rng(d).integers(20, 3000, size=40), [1 << 21, (1 << 21) + 5, 1 << 21]])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(off[-1])
    assert n > LARGE
    g = DyCuckooGroup((sizes / 0.85).astype(np.uint64) + 32, subtables=d, insert_order=0,
                      kick_bound=kick_bound)
    for seed in range(5):
        k = keys(0, n, 11 + seed)
        g.clear()
        g.insert(k, k ^ seed, off)
        v, h = g.find(k, off)
        assert last_rule(g) == START
        assert bool(h.all()) and torch.equal(v, k ^ seed)
    g.close()
