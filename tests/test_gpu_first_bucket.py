"""Finds that rely on the table's first-bucket rule (2^22 lookups or more on a table that nothing was
erased from, resized or loaded since it was empty) against the same lookups in smaller calls, which
read in the reference order: values and flags bit for bit, also for copies of one key in both its
buckets, under each rule and under none, and where an erase on another stream, a captured find or
a refill could leave the rule behind."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LARGE = 1 << 22


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


def both_ways(t, q):
    """The large find, checked against small ones."""
    v, h = t.find(q)
    sv, sh = zip(*(t.find(x) for x in torch.split(q, LARGE - 1)))
    assert torch.equal(h, torch.cat(sh)) and torch.equal(v, torch.cat(sv))
    return v, h


@pytest.mark.parametrize("d", [2, 4, 6])
@pytest.mark.parametrize("order", [0, 3])
def test_same_as_the_reference_order(D, order, d):
    print(f"\n[gpu-case] first-bucket rule d={d} insert_order={order}", flush=True)
    m = 1 << 19
    t = D.DyCuckoo(int(m / (0.6 if d == 2 else 0.75)), subtables=d, insert_order=order, kick_bound=0, auto_resize=0)
    k = keys(0, m)
    q = lookups(LARGE + 77, m, d)
    _, h = both_ways(t, q)  # empty
    assert not h.any()
    t.insert(k, k ^ 1)
    _, h = both_ways(t, q)
    # a second copy of some keys: where the first bucket is full, in the other one
    t.insert(k[: m // 16], k[: m // 16] ^ 2)
    both_ways(t, q)
    # entries under the other rule (a bulk fill into an eviction-built table, or the reverse)
    t.configure(insert_order=3 - order)
    extra = keys(3 * m, 3 * m + m // 32)
    t.insert(extra, extra)
    both_ways(t, torch.cat([q, extra]))
    # erased slots: the rule is gone
    gone = t.erase(k[: m // 2])
    assert gone.all()
    _, h2 = both_ways(t, q)
    assert int(h2.sum()) < int(h.sum())
    t.insert(k[: m // 2], k[: m // 2] ^ 3)
    both_ways(t, q)
    # emptied and filled again: the rule is back
    t.clear()
    t.insert(k, k ^ 4)
    v, h = both_ways(t, q)
    t.resize_up()
    v2, h2 = both_ways(t, q)
    assert torch.equal(h, h2) and torch.equal(v, v2)
    assert t.resize_down()
    both_ways(t, q)
    t.load(t.dump())
    both_ways(t, q)
    t.close()


@pytest.mark.parametrize("d", [2, 4])
@pytest.mark.parametrize("order", [0, 3])
def test_wide_tables(D, order, d):
    print(f"\n[gpu-case] first-bucket rule, wide d={d} insert_order={order}", flush=True)
    m = 1 << 19
    t = D.DyCuckooWide(int(m / (0.6 if d == 2 else 0.75)), subtables=d, insert_order=order, kick_bound=0, auto_resize=0)
    wide = lambda x: x.long() * 0x1_0000_0001 ^ 0x55  # noqa: E731
    k = wide(keys(0, m))
    q = torch.cat([wide(lookups(LARGE + 5, m, d)), torch.tensor([0, -1], device="cuda")])
    _, h = both_ways(t, q)
    assert not h.any()
    t.insert(k, k ^ 1)
    both_ways(t, q)
    t.insert(k[: m // 16], k[: m // 16] ^ 2)
    both_ways(t, q)
    t.upsert(k[: m // 16], k[: m // 16] ^ 3)  # under the start rule
    both_ways(t, q)
    assert t.erase(k[: m // 2]).all()
    both_ways(t, q)
    t.clear()
    t.insert(k, k ^ 4)
    v, h = both_ways(t, q)
    t.resize_up()
    v2, h2 = both_ways(t, q)
    assert torch.equal(h, h2) and torch.equal(v, v2)
    t.close()


def test_upsert_and_host_inserts_keep_the_start_rule(D):
    print("\n[gpu-case] first-bucket rule, upsert and host inserts", flush=True)
    m = 1 << 19
    t = D.DyCuckoo(int(m / 0.8), insert_order=0, kick_bound=15, auto_resize=0)
    k = keys(0, m)
    q = lookups(LARGE, m)
    t.upsert(k[: m // 4], k[: m // 4])
    t.insert_host(k[m // 4: m // 2].cpu().numpy(), k[m // 4: m // 2].cpu().numpy())
    t.insert_async(k[m // 2:], k[m // 2:])
    t.upsert(k[: m // 4], k[: m // 4] ^ 9)
    both_ways(t, q)
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
        gone = t.erase(go, stream=b)
        torch.cuda.synchronize()
        assert gone.all() and h.all() and torch.equal(v, q ^ 5)
        v, h = both_ways(t, k.repeat(4))
        assert torch.equal(h.view(4, m)[0].bool(), torch.arange(m, device="cuda") < m // 2)
    t.close()


def test_captured_find_is_replayed_after_an_erase(D):
    print("\n[gpu-case] first-bucket rule, captured find", flush=True)
    m = 1 << 19
    k = keys(0, m)
    q = lookups(LARGE, m)
    t = D.DyCuckoo(int(m / 0.9), insert_order=3, kick_bound=0, auto_resize=0)
    t.insert(k, k)
    v = torch.empty_like(q)
    h = torch.empty(q.numel(), dtype=torch.uint8, device="cuda")
    t.find(q, v, h)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        t.find(q, v, h)
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
    # a mean of 1 MiB and more a table, from which a group's finds rely on the rule
    sizes = np.random.default_rng(1).integers(0, 400_000, size=24)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(off[-1])
    assert n > LARGE
    k = keys(0, n)
    miss = torch.rand(n, device="cuda") < 0.5
    q = torch.where(miss, keys(n, 2 * n), k)
    if bits == 64:
        k, q = k.long() * 0x9E3779B1 | 1, q.long() * 0x9E3779B1 | 1
    g = (DyCuckooGroup if bits == 32 else DyCuckooWideGroup)((sizes / 0.85).astype(np.uint64) + 128,
                                                             insert_order=order, kick_bound=0)

    def halves():
        cut = sizes.size // 2
        zero = np.zeros(sizes.size - cut, dtype=np.uint64)
        lo = np.concatenate([off[: cut + 1], off[cut] + zero])
        hi = np.concatenate([np.zeros(cut, dtype=np.uint64), off[cut:] - off[cut]])
        c = int(off[cut])
        a, b = g.find(q[:c].contiguous(), lo), g.find(q[c:].contiguous(), hi)
        return torch.cat([a[0], b[0]]), torch.cat([a[1], b[1]])

    for step in range(3):
        if step == 2:
            g.clear()
        if step != 1:
            g.insert(k, k ^ step, off)
        else:
            erased = torch.arange(n, device="cuda") % 3 == 0
            g.erase(torch.where(erased, k, torch.zeros_like(k)), off)
        v, h = g.find(q, off)
        sv, sh = halves()
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
        miss = torch.rand(n, device="cuda") < 0.4
        q = torch.where(miss, keys(n, 2 * n), k)
        g = DyCuckooGroup((sizes / 0.85).astype(np.uint64) + 128, insert_order=order, kick_bound=0)
        p = g.plan(k, k ^ 7, off, q, off)
        for _ in range(3):
            p.run()
            assert torch.equal(p.out_hit.bool(), ~miss)
            assert torch.equal(p.out_vals, torch.where(miss, torch.zeros_like(k), k ^ 7))
            g.erase(k, off)  # eager work between the replays
        g.close()


@pytest.mark.parametrize("d", [2, 4])
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
    g = DyCuckooGroup((sizes / (0.75 if d == 2 else 0.85)).astype(np.uint64) + 32, subtables=d, insert_order=0,
                      kick_bound=kick_bound)
    for seed in range(5):
        k = keys(0, n, 11 + seed)
        g.clear()
        g.insert(k, k ^ seed, off)
        v, h = g.find(k, off)
        assert bool(h.all()) and torch.equal(v, k ^ seed)
    g.close()
