"""Group calls whose items are shared tile by tile among a workgroup's waves: tables of batch sizes
around a tile (64) and around a workgroup's share of tiles, empty tables between them, item sizes
from one tile up, and batches below and above the size where finds are laid out by XCD. Every
find, erase and count is compared exactly with what was put in (32-bit and wide groups)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import databases_gpu_amd as D

    D.load()
    return D


SIZES = [0, 1, 63, 64, 65, 511, 512, 513, 0, 2000, 4095, 4096, 4097, 5000, 3, 0]


def batch(bits, reps, seed):
    """Tables of SIZES, reps times over: distinct keys, values, offsets, and as many lookups, about
    half of them keys of the same table, the rest of its neighbour or of no table."""
    sizes = np.array(SIZES * reps, dtype=np.int64)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(off[-1])
    rng = np.random.default_rng(seed)
    k = rng.permutation(np.arange(1, 2 * n + 1, dtype=np.uint64)) * np.uint64(2654435761)
    k = k % np.uint64(2**32 - 1) if bits == 32 else k * np.uint64(0x9E3779B97F4A7C15)
    k = np.unique(k[(k != 0) & (k < np.uint64(2**64 - 1))])
    rng.shuffle(k)
    keys, absent = k[:n], k[n:]
    vals = (keys ^ np.uint64(0x5bd1e995)) & np.uint64(2**bits - 1)
    q = keys.copy()
    pick = rng.random(n)
    q[pick < 0.3] = rng.choice(absent, size=int((pick < 0.3).sum()))
    q[pick > 0.8] = np.roll(keys, 777)[pick > 0.8]  # keys of another table (or another place of this one)
    owner = np.repeat(np.arange(sizes.size), sizes)
    table_of = dict(zip(keys.tolist(), owner.tolist()))
    hit = np.array([table_of.get(int(x), -1) == t for x, t in zip(q, owner)])
    want = np.where(hit, (q ^ np.uint64(0x5bd1e995)) & np.uint64(2**bits - 1), np.uint64(0))
    return sizes, off, keys, vals, q, hit, want


def dev(a, bits):
    a = a.astype(np.uint32).view(np.int32) if bits == 32 else np.ascontiguousarray(a).view(np.int64)
    return torch.from_numpy(a).cuda()


@pytest.mark.parametrize("item_keys", [64, 500, 4096])
@pytest.mark.parametrize("bits", [32, 64])
def test_sizes_around_tiles(D, bits, item_keys):
    from databases_gpu_amd.table import DyCuckooGroup, DyCuckooWideGroup

    print(f"\n[gpu-case] group tiles bits={bits} item_keys={item_keys}", flush=True)
    sizes, off, keys, vals, q, hit, want = batch(bits, 3, 11 + bits)
    g = (DyCuckooGroup if bits == 32 else DyCuckooWideGroup)((sizes / 0.7).astype(np.uint64) + 128, kick_bound=0)
    if bits == 32:
        g.set_launch(item_keys=item_keys)
    g.insert(dev(keys, bits), dev(vals, bits), off)
    u = np.uint32 if bits == 32 else np.uint64
    for _ in range(2):
        v, h = g.find(dev(q, bits), off)
        assert np.array_equal(h.cpu().numpy().astype(bool), hit)
        assert np.array_equal(v.cpu().numpy().view(u), want.astype(u))
    assert [g.table_stats(i)["count"] for i in range(sizes.size)] == sizes.tolist()
    gone = g.erase(dev(q, bits), off).cpu().numpy().astype(bool)
    assert not (gone & ~hit).any()
    deleted = {}  # a key asked for twice in its table is deleted once
    for x, d in zip(q[hit].tolist(), gone[hit].tolist()):
        deleted[x] = deleted.get(x, 0) + d
    assert all(c == 1 for c in deleted.values())
    counts = sizes.copy()
    np.subtract.at(counts, np.repeat(np.arange(sizes.size), sizes)[gone], 1)
    assert [g.table_stats(i)["count"] for i in range(sizes.size)] == counts.tolist()
    _, h = g.find(dev(q, bits), off)
    assert not h.cpu().numpy().any()
    g.close()


@pytest.mark.parametrize("kick_bound", [0, 15])
@pytest.mark.parametrize("item_keys", [0, 64, 500])
@pytest.mark.parametrize("n", [(1 << 16) - 1, 1 << 16, 400_000])
def test_inserts_of_shared_and_of_whole_items(D, n, item_keys, kick_bound):
    """Below 2^16 keys the waves of a workgroup share an insert's items, from there on each takes whole
    ones: tables of sizes around a tile and around an item, full ones among them."""
    from databases_gpu_amd.table import DyCuckooGroup
    from databases_gpu_amd.workload import keys_range, splitmix32

    print(f"\n[gpu-case] group insert of {n} keys, item_keys={item_keys} kick_bound={kick_bound}", flush=True)
    sizes = np.array(SIZES * (n // sum(SIZES)) + [0], dtype=np.int64)
    sizes[-1] = n - sizes.sum()
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    dv = torch.device("cuda", 0)
    k = keys_range(0, n, 21, dv)
    g = DyCuckooGroup((sizes / 0.85).astype(np.uint64) + 32, insert_order=0, kick_bound=kick_bound)
    g.set_launch(item_keys=item_keys)
    miss = torch.rand(n, device=dv) < 0.4
    q = torch.where(miss, keys_range(n, 2 * n, 21, dv), k)
    for _ in range(2):
        g.clear()
        g.insert(k, splitmix32(k), off)
        assert [g.table_stats(i)["count"] for i in range(sizes.size)] == sizes.tolist()
        v, h = g.find(q, off)
        assert torch.equal(h.bool(), ~miss)
        assert torch.equal(v, torch.where(miss, torch.zeros_like(k), splitmix32(k)))
    g.close()


@pytest.mark.parametrize("order", [0, 3])
def test_large_find_is_laid_out_by_xcd(D, order):
    """More than 2^22 lookups: items on their tables' XCDs, empty places among them."""
    from databases_gpu_amd.table import DyCuckooGroup

    print(f"\n[gpu-case] group find of 2^22 keys, insert_order={order}", flush=True)
    from databases_gpu_amd.workload import keys_range, splitmix32

    rng = np.random.default_rng(5)
    sizes = rng.integers(0, 40_000, size=230)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(off[-1])
    assert n > 1 << 22
    dv = torch.device("cuda", 0)
    k = keys_range(0, n, 9, dv)
    g = DyCuckooGroup((sizes / 0.8).astype(np.uint64) + 128, insert_order=order, kick_bound=0)
    g.insert(k, splitmix32(k), off)
    miss = torch.rand(n, device=dv) < 0.4
    q = torch.where(miss, keys_range(n, 2 * n, 9, dv), k)
    v, h = g.find(q, off)
    assert torch.equal(h.bool(), ~miss)
    assert torch.equal(v, torch.where(miss, torch.zeros_like(k), splitmix32(k)))
    g.close()
