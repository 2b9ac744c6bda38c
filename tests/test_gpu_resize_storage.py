"""Resizes that take the storage an earlier one left: up and down around one size, up twice (the kept
block has the wrong size), finds on a second stream in between (nothing is kept then), and blocks
above the bound; every key is found after each step and the memory in use stays bounded."""
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


def table(D, bits, capacity):
    from databases_gpu_amd.table import DyCuckooWide

    return (DyCuckooWide if bits == 64 else D.DyCuckoo)(capacity, auto_resize=0)


def contents(bits, n):
    from databases_gpu_amd.workload import keys_range, u32_to_i64

    k = keys_range(0, 2 * n, 9, torch.device("cuda", 0))
    k = u32_to_i64(k) if bits == 64 else k
    return k[:n], k


def check(t, k, q, stream):
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        v, h = t.find(q)
    torch.cuda.synchronize()
    assert bool(h[: k.numel()].all()) and not bool(h[k.numel():].any())
    assert torch.equal(v[: k.numel()], k ^ 77)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("second_stream", [False, True])
@pytest.mark.parametrize("capacity", [1 << 12, 3 << 18, 9 << 23])
def test_resizes_in_turn(D, bits, second_stream, capacity):
    print(f"\n[gpu-case] resizes in turn, {bits} bits, {capacity} slots, second stream {second_stream}", flush=True)
    t = table(D, bits, capacity)
    own = torch.cuda.current_stream()
    other = torch.cuda.Stream() if second_stream else own
    k, q = contents(bits, min(capacity // 2, 1 << 20))
    t.insert(k, k ^ 77)
    torch.cuda.synchronize()
    size = t.stats()["capacity"] * bits // 4
    used = []
    for step in "ududuuddud":
        if step == "u":
            t.resize_up()
        else:
            assert t.resize_down()
        check(t, k, q, other if step == "u" else own)
        used.append(torch.cuda.mem_get_info()[0])
    assert t.stats()["count"] == k.numel()
    # the table itself, at most one and a half times its first size, a kept block and frees not yet done
    assert max(used) - min(used) < 2 * size + (512 << 20)
    t.close()
