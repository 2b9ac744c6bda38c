"""The insert's lanes and quads where they can go wrong: ragged batches around a wave's chunk of 64
entries, more copies of one key than a bucket's slots (lost races on one bucket), nearly full
tables, both eviction rules (kick_bound 15 and 0) and reserved keys. The stored multiset, the
placement invariant, the counters and the finds are compared with the batch and the oracle."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import databases_gpu_amd as D

    D.load()
    return D


def distinct(n, seed):
    rng = np.random.default_rng(seed)
    out = np.unique(rng.integers(1, 2**32 - 1, size=2 * n + 64, dtype=np.uint64).astype(np.uint32))
    rng.shuffle(out)
    return out[:n]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


@pytest.mark.parametrize("kick_bound", [0, 15])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1023])
@pytest.mark.parametrize("d", [2, 4, 6])
def test_ragged_batches_with_copies(D, n, d, kick_bound):
    print(f"\n[gpu-case] insert n={n} d={d} kick_bound={kick_bound}", flush=True)
    rng = np.random.default_rng(n + d)
    keys = distinct(n, 7 * n + d)
    if n > 60:
        keys[:20] = keys[0]  # 20 copies of one key: more than a bucket holds
        keys[n // 2] = 0
        keys[-1] = 0xFFFFFFFF
    keys = rng.permutation(keys)
    vals = np.arange(1, n + 1, dtype=np.uint32) * np.uint32(2654435761)
    t = D.DyCuckoo(max(64, int(n / 0.8)), subtables=d, kick_bound=kick_bound, auto_resize=0)
    t.insert(dev(keys), dev(vals))
    ok = (keys != 0) & (keys != 0xFFFFFFFF)
    st = t.stats()
    assert st["rejected"] == n - ok.sum() and st["count"] == ok.sum() and st["lost"] == 0
    img = t.dump()
    stored = np.concatenate(img)
    stored = np.sort(np.concatenate([stored[stored != 0], t.pending()]))
    want = np.sort((keys[ok].astype(np.uint64) << np.uint64(32)) | vals[ok])
    assert np.array_equal(stored, want)
    ref = O.OracleTable(nb=t.buckets)
    ref.sub = [x.copy() for x in img]
    assert ref.check_invariant() == 0
    _, h = t.find(dev(keys))
    assert np.array_equal(h.cpu().numpy(), ok.astype(np.uint8))
    t.close()


@pytest.mark.parametrize("kick_bound", [0, 15])
def test_batch_to_a_nearly_full_table(D, kick_bound):
    """Fill 0.97 in several batches: most chains evict, and every key is found."""
    print(f"\n[gpu-case] insert to fill 0.97, kick_bound={kick_bound}", flush=True)
    t = D.DyCuckoo(1 << 16, kick_bound=kick_bound, auto_resize=0, max_fail_rounds=0)
    keys = distinct(int(t.capacity * 0.97), 5 + kick_bound)
    vals = keys ^ np.uint32(0xA5A5A5A5)
    for part in np.array_split(np.arange(keys.size), 5):
        try:
            t.insert(dev(keys[part]), dev(vals[part]))
        except D.DycError:
            pass  # entries past the eviction bound wait on the pending list
    v, h = t.find(dev(keys))
    assert h.cpu().numpy().all() and np.array_equal(v.cpu().numpy().view(np.uint32), vals)
    assert t.stats()["count"] == keys.size
    t.close()
