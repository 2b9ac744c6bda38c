"""The launch-shape autotuner's choices (databases_gpu_amd/autotune.py) without a GPU, over stand-ins
for a group and a table whose calls take a time that depends on the shape set last."""
import json

import numpy as np
import pytest
import torch

from databases_gpu_amd import autotune


class Fake:
    """A group or a table: remembers the shape set last, and every shape a call ran with."""

    device = torch.device("cpu")
    capacity = 1 << 12

    def __init__(self, **shape):
        self.shape = dict(shape)
        self.ran = {"insert": [], "find": []}
        self.last = None

    def set_launch(self, **shape):
        self.shape.update(shape)

    configure = set_launch

    def config(self):
        return dict(self.shape)

    def clear(self, stream=None):
        pass

    def insert(self, *a):
        self.last = "insert"
        self.ran["insert"].append(dict(self.shape))

    def find(self, *a):
        self.last = "find"
        self.ran["find"].append(dict(self.shape))


@pytest.fixture
def timed(monkeypatch, tmp_path):
    """cost[op](shape) is what a timed call of op takes."""
    cost = {"insert": lambda s: 1.0, "find": lambda s: 1.0}
    holder = {}

    def run(fn, reps):
        fn()
        t = holder["t"]
        return cost[t.last](t.shape)

    monkeypatch.setattr(autotune, "_time", run)
    monkeypatch.setattr(autotune, "CACHE_PATH", str(tmp_path / "cache.json"))
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda d: "gpu")
    return holder, cost


def tune(holder, kind, **kw):
    keys = torch.arange(1, 4097, dtype=torch.int32)
    if kind == "group":
        t = Fake(find_lanes=8, insert_lanes=1, find_blocks=0, insert_blocks=0, item_keys=4096, kick_bound=15)
        holder["t"] = t
        off = np.array([0, 1024, 4096], dtype=np.uint64)
        return t, autotune.tune_group(t, keys, keys, off, keys, off, reps=1, **kw)
    t = Fake(find_lanes=8, insert_lanes=1, max_blocks=kw.pop("max_blocks", 0), insert_blocks=0, kick_bound=15,
             block_threads=256)
    holder["t"] = t
    return t, autotune.tune_table(t, keys, keys, keys, reps=1, **kw)


@pytest.mark.parametrize("kind", ["group", "table"])
def test_no_shape_is_timed_twice_and_lanes_are_left_alone(timed, kind):
    holder, _ = timed
    t, out = tune(holder, kind, use_cache=False)
    for op in ("insert", "find"):
        seen = {json.dumps(s, sort_keys=True) for s in t.ran[op]}
        # an insert trial runs once untimed before it is timed, and once more with the chosen shape
        runs = 2 if op == "insert" else 1
        assert len(t.ran[op]) <= runs * len(seen) + 1
        assert {s["find_lanes"] for s in t.ran[op]} == {8} and {s["insert_lanes"] for s in t.ran[op]} == {1}
    # all equal: the library's defaults
    assert out["installed"]["insert_blocks"] == 0
    assert out["installed"].get("find_blocks", 0) == 0 and out["installed"].get("max_blocks", 0) == 0


@pytest.mark.parametrize("best", [0, 512, 1024])
def test_a_group_gets_the_grid_that_is_fastest(timed, best):
    """512 workgroups, the library's own choice from 2^24 keys on, and its default are candidates."""
    holder, cost = timed
    cost["find"] = lambda s: 1.0 if s["find_blocks"] == best else 2.0
    t, out = tune(holder, "group", use_cache=False)
    assert out["installed"]["find_blocks"] == best == t.shape["find_blocks"]
    # the find is timed at the item size that is installed
    assert {s["item_keys"] for s in t.ran["find"]} == {t.shape["item_keys"]}


def test_a_capped_find_grid_stays_capped(timed):
    holder, _ = timed
    t, out = tune(holder, "table", use_cache=False, max_blocks=77)
    assert out["installed"]["max_blocks"] == 77 and {s["max_blocks"] for s in t.ran["find"]} == {77}


@pytest.mark.parametrize("kind", ["group", "table"])
def test_shapes_cached_for_other_kernels_are_not_installed(timed, kind):
    holder, _ = timed
    _, out = tune(holder, kind)
    with open(autotune.CACHE_PATH) as f:
        cache = json.load(f)
    (key,) = cache
    # as this version cached it: reused
    _, again = tune(holder, kind)
    assert again["installed"] == out["installed"] and not holder["t"].ran["insert"]
    # as the kernels before it did: without a version, and with another one
    for old in (key.replace(f"|v{autotune.SHAPES}", ""), key.replace(f"|v{autotune.SHAPES}", f"|v{autotune.SHAPES - 1}")):
        assert old != key
        with open(autotune.CACHE_PATH, "w") as f:
            json.dump({old: {"insert": {"insert_blocks": 7, "ms": 1.0}, "find": {"ms": 1.0}, "trials": 1}}, f)
        _, new = tune(holder, kind)
        assert new["installed"]["insert_blocks"] != 7 and holder["t"].ran["insert"]
