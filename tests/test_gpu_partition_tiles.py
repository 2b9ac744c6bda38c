"""Bulk inserts at the sizes where the partition's tiles change or end: one entry to a few tiles, the
batches on both sides of the larger tiles' rule, and those a tile and a block range do not divide;
every key is found with its value, and nothing else is."""
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


def keys(lo, hi, seed=5):
    from databases_gpu_amd.workload import keys_range

    return keys_range(lo, hi, seed, torch.device("cuda", 0))


TILE = 4096
CASES = [  # keys the table is sized for, entries of the batch
    (1 << 18, 1), (1 << 18, TILE - 1), (1 << 18, TILE), (1 << 18, TILE + 1), (1 << 20, 3 * TILE + 77),
    (3 << 20, 1 << 21), (20 << 20, (1 << 24) - 1), (20 << 20, 1 << 24), (20 << 20, (1 << 24) + 14337),
    (70 << 20, (1 << 26) - 1), (70 << 20, (1 << 26) + 12289),
    # more than 2^16 chunks: 4-byte chunk ids, three passes
    (456 << 20, (3 << 20) + 1), (456 << 20, (1 << 24) + 5),
]


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("sized, n", CASES)
def test_every_key_of_a_bulk_insert_is_found(D, bits, sized, n):
    print(f"\n[gpu-case] bulk insert of {n} keys of {bits} bits into a table for {sized}", flush=True)
    if bits == 64:
        from databases_gpu_amd.table import DyCuckooWide
        from databases_gpu_amd.workload import u32_to_i64

        t = DyCuckooWide(int(sized / 0.85), insert_order=3, kick_bound=0)
        k, other = (u32_to_i64(keys(*r)) * 0x1_0000_0001 for r in ((0, n), (n, n + 4096)))
    else:
        t = D.DyCuckoo(int(sized / 0.85), insert_order=3, kick_bound=0)
        k, other = keys(0, n), keys(n, n + 4096)
    v = k ^ 0x5A5A
    t.insert(k, v)
    s = t.stats()
    assert s["count"] == n and s["pending"] == 0 and s["lost"] == 0
    got, hit = t.find(k)
    assert hit.all() and torch.equal(got, v)
    assert not t.find(other)[1].any()
