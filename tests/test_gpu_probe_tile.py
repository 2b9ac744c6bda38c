"""The probe tile (find, erase, update) where it can go wrong: ragged tails, reserved keys among
the lookups, and copies of one key in several slots of one lane's part of a bucket, in several
lanes' parts, and in both buckets of its pair. Everything is compared exactly with the oracle on
the oracle's own images, whatever lanes per key the table asks for."""
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


def images_with_copies(seed, d):
    """Oracle images of distinct keys, 24 of them with 2..32 copies (values tell copies apart)."""
    rng = np.random.default_rng(seed)
    keys = distinct(600, seed)
    reps = np.ones(keys.size, dtype=np.int64)
    reps[:24] = rng.integers(2, 33, size=24)
    batch = rng.permutation(np.repeat(keys, reps))
    vals = np.arange(1, batch.size + 1, dtype=np.uint32) * np.uint32(2654435761)
    tb = O.OracleTable(nb=[32 if d == 2 else 16] * d, rescue_kicks=128, max_fail_rounds=0)
    tb.insert(batch, vals)  # copies that fit neither bucket stay pending, outside the images
    return [np.ascontiguousarray(x).copy() for x in tb.images()], keys


def on_oracle(images):
    tb = O.OracleTable(nb=[x.size // 16 for x in images])
    tb.sub = [x.copy() for x in images]
    return tb


@pytest.mark.parametrize("d", [2, 4, 6])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 130, 601])
def test_find_erase_update_with_copies(D, d, n):
    print(f"\n[gpu-case] probe tile d={d} n={n}", flush=True)
    images, keys = images_with_copies(40 + d, d)
    absent = distinct(900, 77)
    absent = absent[~np.isin(absent, keys)][:200]
    rng = np.random.default_rng(n)
    q = np.concatenate([keys[:400], absent, np.array([0], dtype=np.uint32)])
    q = rng.permutation(q)[:n] if n > 1 else keys[:1]
    t = D.DyCuckoo(1000, subtables=d, max_fail_rounds=0, find_lanes=[4, 8, 16][n % 3])
    t.load(images)
    v, h = t.find(dev(q))
    want_v, want_h = on_oracle(images).find(q)
    assert np.array_equal(h.cpu().numpy(), want_h)
    assert np.array_equal(v.cpu().numpy().view(np.uint32), want_v)
    # update rewrites, and erase empties, every copy in the bucket that find reads, and no other
    ref = on_oracle(images)
    flags = ref.erase(q)
    erased = ref.images()
    u = q[flags != 0]
    if u.size:
        new = u ^ np.uint32(0x5bd1e995)
        assert t.upsert(dev(u), dev(new)).cpu().numpy().all()
        for got, old, gone in zip(t.dump(), images, erased):
            want = old.copy()
            hit = old != gone
            k = want[hit] >> np.uint64(32)
            want[hit] = (k << np.uint64(32)) | (k ^ np.uint64(0x5bd1e995))
            assert np.array_equal(got, want)
    assert np.array_equal(t.erase(dev(q)).cpu().numpy(), flags)
    assert all(np.array_equal(a, b) for a, b in zip(t.dump(), erased))
    t.close()


@pytest.mark.parametrize("d", [2, 4])
@pytest.mark.parametrize("n", [1, 64, 65, 601])
def test_wide_find_erase_update_with_copies(D, d, n):
    """The wide probe over the same images: keys below 2^32 live where the 32-bit table puts them."""
    print(f"\n[gpu-case] wide probe tile d={d} n={n}", flush=True)
    images, keys = images_with_copies(40 + d, d)
    absent = distinct(900, 77)
    absent = absent[~np.isin(absent, keys)][:200]
    rng = np.random.default_rng(n)
    q = np.concatenate([keys[:400], absent, np.array([0], dtype=np.uint32)])
    q = rng.permutation(q)[:n] if n > 1 else keys[:1]
    wide = lambda a: torch.from_numpy(a.astype(np.uint64).view(np.int64)).cuda()  # noqa: E731
    lo = np.uint64(0xFFFFFFFF)
    t = D.DyCuckooWide(1000, subtables=d, max_fail_rounds=0)
    t.load([x >> np.uint64(32) for x in images], [x & lo for x in images])
    v, h = t.find(wide(q))
    want_v, want_h = on_oracle(images).find(q)
    assert np.array_equal(h.cpu().numpy(), want_h)
    assert np.array_equal(v.cpu().numpy().view(np.uint64), want_v.astype(np.uint64))
    ref = on_oracle(images)
    flags = ref.erase(q)
    u = q[flags != 0]
    if u.size:
        new = u.astype(np.uint64) * np.uint64(0x100000001)
        assert t.upsert(wide(u), torch.from_numpy(new.view(np.int64)).cuda()).cpu().numpy().all()
        gk, gv = t.dump()
        for k, val, old, gone in zip(gk, gv, images, ref.images()):
            hit = old != gone
            assert np.array_equal(k, old >> np.uint64(32))
            assert np.array_equal(val, np.where(hit, (old >> np.uint64(32)) * np.uint64(0x100000001), old & lo))
    # erase empties the key words of every copy in the bucket that find reads, and no other
    assert np.array_equal(t.erase(wide(q)).cpu().numpy(), flags)
    for k, gone in zip(t.dump()[0], ref.images()):
        assert np.array_equal(k, gone >> np.uint64(32))
    t.close()
