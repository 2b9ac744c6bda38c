"""The work a user has this library do, as cases that can be timed.

Each case is one pass through the public entry points (``databases_gpu_amd``): loading a table and
looking keys up in it, a stream's batches against a live table, tables of many sizes in one call,
host arrays, queued requests. ``listed()`` gives the fixed cases, ``draw()`` more of the same
ranges. Every output is a stored value, a flag or a count, so results are compared exactly.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import databases_gpu_amd as D
from databases_gpu_amd.server import DyCuckooServer
from databases_gpu_amd.table import DyCuckooGroup, DyCuckooWide, DyCuckooWideGroup, HashAPI
from databases_gpu_amd.workload import keys_range, splitmix32, u32_to_i64

# What every case holds: kind (below), bits of a key (32 or 64), keys stored before the pass or
# loaded by it, n (the pass's batch), d (subtables), theta (fill after loading), hit (share of
# lookups that are stored) and the table options in earnest use.
_COMMON = {"bits": 32, "d": 4, "theta": 0.9, "hit": 0.5, "order": 3, "kick_bound": 0, "find_lanes": 4}


def _case(name=None, **fields):
    c = dict(_COMMON, **fields)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a lookup call of a few keys: an index probe in a query, where latency counts
        _case("find_small", kind="find", keys=1 << 16, n=1021, order=0, kick_bound=15, find_lanes=8),
        # the headline: build a 2^28-key table by bulk insert, then uniform and Zipf lookups
        _case("load_u32_2p28", kind="load", keys=1 << 28, n=1 << 28, zipf=True),
        # an ordinary build and probe side (join, group-by) with the library's default options
        _case("load_u32_default", kind="load", keys=5_000_011, n=5_000_011, theta=0.85, hit=0.6, order=0,
              kick_bound=15, find_lanes=8, zipf=False),
        # the same with 64-bit keys and values
        _case("load_u64_2p26", kind="load", bits=64, keys=1 << 26, n=1 << 26, zipf=False),
        # one batch of a dynamic stream: insert fresh keys, look up, delete
        _case("churn_u32", kind="churn", keys=1 << 25, n=1_677_721, theta=0.8, hit=0.7, order=0),
        # the smallest stream batches, where each call's launches and wait are the cost
        _case("churn_small", kind="churn", keys=1 << 20, n=1000, theta=0.8, hit=0.7, order=0),
        # insert-or-update of a batch of which half is stored already
        _case("upsert_u32", kind="upsert", keys=1 << 23, n=(1 << 20) + 7, theta=0.75, hit=0.5, order=0),
        # a table that grows and shrinks by one subtable, looked up at each size
        _case("resize_u32", kind="resize", keys=1 << 24, n=1 << 20, theta=0.7, hit=0.5, order=0),
        # thousands of uneven tables built and probed in one call each
        _case("group_u32", kind="group", tables=2048, lo=8, hi=18, theta=0.85, hit=0.6),
        # a small step over many little tables, captured once and replayed
        _case("group_plan", kind="plan", tables=256, lo=4, hi=8, theta=0.85, hit=0.6, order=0),
        # the reference's host-array calls, transfers included
        _case("host_u32", kind="host", keys=1 << 22, n=(1 << 22) + 12_345, theta=0.45, hit=0.5, order=0,
              kick_bound=15, find_lanes=8),
        # queued requests of many tenants, served together
        _case("serve_u32", kind="serve", tables=64, lo=6, hi=14, theta=0.8, hit=0.5, order=0),
    ]


def _logint(rng, lo, hi):
    """An integer in [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["find", "load", "load", "churn", "churn", "upsert", "resize", "group", "plan", "host", "serve"])
    c = _case(kind=kind, d=rng.choice([2, 3, 4, 4, 4, 5, 6]), hit=round(rng.uniform(0.1, 1.0), 2),
              kick_bound=rng.choice([0, 15]), find_lanes=rng.choice([4, 8, 16]))
    if kind == "find":
        c.update(keys=_logint(rng, 1 << 12, 1 << 25), n=_logint(rng, 1, 1 << 25), theta=0.8, order=rng.choice([0, 3]))
    elif kind == "load":
        c.update(bits=rng.choice([32, 32, 64]), order=rng.choice([0, 3, 3]), theta=round(rng.uniform(0.5, 0.9), 2),
                 zipf=rng.random() < 0.3)
        c.update(keys=_logint(rng, 1 << 12, 1 << (27 if c["bits"] == 32 else 26)))
        c.update(n=max(1, int(c["keys"] * rng.uniform(0.25, 1.0))))
        if c["d"] == 2:
            c["theta"] = min(c["theta"], 0.8)
    elif kind in ("churn", "upsert"):
        c.update(bits=rng.choice([32, 32, 64]), keys=_logint(rng, 1 << 14, 1 << 25), theta=0.75, order=0)
        c.update(n=_logint(rng, 64, max(64, c["keys"] // 16)))
    elif kind == "resize":
        c.update(keys=_logint(rng, 1 << 14, 1 << 25), theta=0.7, order=0)
        c.update(n=_logint(rng, 1 << 10, 1 << 21))
    elif kind == "group":
        hi = rng.randint(9, 18)
        c.update(bits=rng.choice([32, 32, 64]), tables=_logint(rng, 16, 2048), lo=rng.randint(4, 8), hi=hi,
                 theta=round(rng.uniform(0.5, 0.85), 2), order=rng.choice([0, 3]))
        if c["d"] == 2:
            c["theta"] = min(c["theta"], 0.75)
    elif kind == "plan":
        c.update(tables=_logint(rng, 16, 1024), lo=rng.randint(3, 6), hi=rng.randint(7, 12),
                 theta=round(rng.uniform(0.5, 0.85), 2), order=rng.choice([0, 3]))
        if c["d"] == 2:
            c["theta"] = min(c["theta"], 0.75)
    elif kind == "host":
        c.update(keys=_logint(rng, 1 << 12, 1 << 23), theta=0.45, order=0)
        c.update(n=max(1, int(c["keys"] * rng.uniform(0.25, 0.9))))
    else:
        c.update(tables=_logint(rng, 4, 256), lo=rng.randint(4, 7), hi=rng.randint(8, 16), theta=0.8, order=0)
    return c


# ------------------------------------------------------------------------------------ inputs
def _gen(seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _wide(k32):
    """64-bit keys from distinct 32-bit ones (the low words stay distinct, none is reserved)."""
    lo = u32_to_i64(k32)
    return (splitmix32(k32).to(torch.int64) << 32) | lo


def _keys(c, lo, hi, seed, dev):
    k = keys_range(lo, hi, seed % 100_003 + 1, dev)
    return _wide(k) if c["bits"] == 64 else k


def _values(c, keys):
    """The value stored with each key (all of 32 or 64 bits)."""
    return keys * -7046029254386353131 + 1442695040888963407 if c["bits"] == 64 else splitmix32(keys)


def _new_values(c, keys):
    return _values(c, keys) ^ 0x2545F491


def _lookups(c, present, n, absent_lo, seed, dev):
    """(lookups, hit flags): each lookup is a random stored key with probability hit, else a key
    that was never stored."""
    g = _gen(seed + 1, dev)
    is_hit = torch.rand(n, generator=g, device=dev) < c["hit"]
    idx = torch.randint(0, present.numel(), (n,), generator=g, device=dev)
    q = torch.where(is_hit, present[idx], _keys(c, absent_lo, absent_lo + n, seed, dev))
    return q, is_hit


def _zipf(present, n, seed, dev):
    """Lookups of stored keys with Zipf(0.99) ranks, by the inverse of the continuous CDF: one
    elementwise formula, so a seed always gives the same lookups (a cumulative sum on the GPU
    rounds differently from run to run)."""
    e, m = 1.0 - 0.99, present.numel()
    u = torch.rand(n, generator=_gen(seed + 2, dev), device=dev, dtype=torch.float64)
    rank = (u.mul_(float(m) ** e - 1.0).add_(1.0)).pow_(1.0 / e).sub_(1.0).long()
    return present[rank.clamp_(0, m - 1)]


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _config(c):
    return {"subtables": c["d"], "insert_order": c["order"], "kick_bound": c["kick_bound"],
            "find_lanes": c["find_lanes"]}


def _table(c, **more):
    hint = int(math.ceil(c["keys"] / c["theta"]))
    return (DyCuckooWide if c["bits"] == 64 else D.DyCuckoo)(hint, **_config(c), **more)


def _table_sizes(c):
    """Key counts of a group's tables, log-uniform in [2^lo, 2^hi] (the case's, whatever the seed)."""
    r = np.random.default_rng((c["tables"], c["lo"], c["hi"]))
    return np.maximum(1, np.exp2(r.uniform(c["lo"], c["hi"], size=c["tables"])).astype(np.int64))


def _inputs(c, seed, dev):
    """The pass's inputs as plain tensors (also what exact() works from)."""
    s = {}
    kind = c["kind"]
    if kind in ("group", "plan", "serve"):
        sizes = _table_sizes(c)
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
        n = int(off[-1])
        s["off"], s["sizes"] = off, sizes
        s["k"] = _keys(c, 0, n, seed, dev)
        s["v"] = _values(c, s["k"])
        g = _gen(seed + 1, dev)
        begin = torch.from_numpy(off[:-1].astype(np.int64)).to(dev)
        size = torch.from_numpy(sizes).to(dev)
        which = torch.repeat_interleave(torch.arange(c["tables"], device=dev), size)
        idx = begin[which] + (torch.rand(n, generator=g, device=dev, dtype=torch.float64) * size[which]).long()
        s["is_hit"] = torch.rand(n, generator=g, device=dev) < c["hit"]
        s["q"] = torch.where(s["is_hit"], s["k"][idx], _keys(c, n, 2 * n, seed, dev))
        return s
    m, n = c["keys"], c["n"]
    s["base"] = _keys(c, 0, m, seed, dev)
    if kind in ("churn", "upsert", "host"):
        s["k"] = _keys(c, m, m + n, seed, dev)  # the batch's fresh keys
        s["q"], s["is_hit"] = _lookups(c, torch.cat([s["base"], s["k"]]), n, m + n, seed, dev)
    else:
        s["q"], s["is_hit"] = _lookups(c, s["base"], n, m, seed, dev)
    if kind == "upsert":  # half of the batch is stored already
        g = _gen(seed + 3, dev)
        old = s["base"][torch.randperm(m, generator=g, device=dev)[: n // 2]]
        s["fresh"] = s["k"][: n - n // 2]
        s["old"] = old
        s["k"] = torch.cat([old, s["fresh"]])[torch.randperm(n, generator=g, device=dev)]
        s["q"], s["is_hit"] = _lookups(c, torch.cat([s["base"], s["fresh"]]), n, m + n, seed, dev)
    if c.get("zipf"):
        s["zq"] = _zipf(s["base"], n, seed, dev)
    return s


# --------------------------------------------------------------------------------- the passes
def prepare(case, seed):
    """Inputs on the device and the handle (table, group, plan, server) a program keeps."""
    c, dev = case, _dev()
    s = _inputs(c, seed, dev)
    s["case"] = c
    kind = c["kind"]
    if kind == "load":
        s["t"] = _table(c)
        s["v"] = _values(c, s["base"])
    elif kind in ("find", "resize", "churn", "upsert"):
        s["t"] = _table(c, **({"auto_resize": 1} if kind == "churn" else {}))
        s["t"].insert(s["base"], _values(c, s["base"]))
        if kind == "churn":
            s["v"] = _values(c, s["k"])
        if kind == "upsert":
            s["v"] = _new_values(c, s["k"])
            s["v_old"] = _values(c, s["old"])
    elif kind in ("group", "plan"):
        hints = np.ceil(s["sizes"] / c["theta"]).astype(np.uint64) + 16 * c["d"]
        cls = DyCuckooWideGroup if c["bits"] == 64 else DyCuckooGroup
        s["t"] = cls(hints, **_config(c))
        if kind == "plan":
            s["plan"] = s["t"].plan(s["k"], s["v"], s["off"], s["q"], s["off"])
    elif kind == "host":
        s["api"] = HashAPI(int(math.ceil(c["keys"] / c["theta"])), **_config(c))
        base = s["base"].cpu().numpy().view(np.uint32)
        s["api"].hash_insert(base, _values(c, s["base"]).cpu().numpy().view(np.uint32), base.size)
        s["hv"] = _values(c, s["k"]).cpu().numpy().view(np.uint32)
        s["hk"] = s["k"].cpu().numpy().view(np.uint32)
        s["hq"] = s["q"].cpu().numpy().view(np.uint32)
        s["ans"] = np.zeros(c["n"], dtype=np.uint32)
        s["del"] = np.zeros(c["n"], dtype=np.uint8)
    else:
        hints = np.ceil(s["sizes"] * 2 / c["theta"]).astype(np.uint64) + 16 * c["d"]
        s["t"] = DyCuckooServer(hints, hbm_budget=1 << 30, **_config(c))
        n = s["q"].numel()
        s["out"] = torch.zeros(n, dtype=torch.int32, device=dev)
        s["hit"] = torch.zeros(n, dtype=torch.uint8, device=dev)
        s["del"] = torch.zeros(n, dtype=torch.uint8, device=dev)
        torch.cuda.synchronize()  # requests take inputs that are complete on the device
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "find":
        return s["t"].find(s["q"])
    if kind == "load":
        t = s["t"]
        t.clear()
        t.insert(s["base"], s["v"])
        out = t.find(s["q"])
        if "zq" in s:
            out = out + t.find(s["zq"])
        return out + (t.stats()["count"],)
    if kind == "churn":
        t = s["t"]
        t.insert(s["k"], s["v"])
        out = t.find(s["q"])
        return out + (t.erase(s["k"]), t.stats()["count"])
    if kind == "upsert":
        t = s["t"]
        up = t.upsert(s["k"], s["v"])
        out = t.find(s["q"])
        gone = t.erase(s["fresh"])
        back = t.upsert(s["old"], s["v_old"])
        return (up,) + out + (gone, back, t.stats()["count"])
    if kind == "resize":
        t = s["t"]
        t.resize_up()
        out = t.find(s["q"])
        t.resize_down()
        return out + t.find(s["q"]) + (t.stats()["count"],)
    if kind == "group":
        t = s["t"]
        t.clear()
        t.insert(s["k"], s["v"], s["off"])
        return t.find(s["q"], s["off"])
    if kind == "plan":
        s["plan"].run()
        return s["plan"].out_vals, s["plan"].out_hit
    if kind == "host":
        api, n = s["api"], c["n"]
        api.hash_insert(s["hk"], s["hv"], n)
        hit = api.hash_search(s["hq"], s["ans"], n)
        api.hash_delete(s["hk"], s["del"], n)
        return s["ans"], hit, s["del"]
    t, off = s["t"], s["off"]
    spans = [slice(int(off[i]), int(off[i + 1])) for i in range(c["tables"])]
    for i, x in enumerate(spans):
        t.insert(i, s["k"][x], s["v"][x])
    for i, x in enumerate(spans):
        t.find(i, s["q"][x], s["out"][x], s["hit"][x])
    for i, x in enumerate(spans):
        t.erase(i, s["k"][x], s["del"][x])
    t.drain()
    return s["out"], s["hit"], s["del"]


# ----------------------------------------------------------------------------- what it must do
def work(case):
    """Bytes of one pass: each input read once, each output written once, and of the table the
    lines that the keys' entries lie in (a 128-byte bucket line a key, up to the whole table)."""
    c = case
    w = c["bits"] // 8
    if c["kind"] in ("group", "plan", "serve"):
        m = n = int(_table_sizes(c).sum())
    else:
        m, n = c["keys"], c["n"]
    line = 128 if w == 4 else 256  # a bucket's slots: 16 entries
    table = int(m / c["theta"] * 2 * w)
    probe = min(table, n * line)
    ins = 2 * w * n + min(table, n * (line + 2 * w))
    find = w * n + (w + 1) * n + probe
    erase = w * n + n + min(table, n * (line + w))
    kind = c["kind"]
    if kind in ("find",):
        b = find
    elif kind in ("load", "group", "plan"):
        b = 2 * w * m + table + find * (2 if c.get("zipf") else 1)
    elif kind == "churn":
        b = ins + find + erase
    elif kind == "upsert":
        b = ins + n + find + erase // 2 + ins // 2
    elif kind == "resize":
        b = 2 * find + 6 * table // c["d"]
    else:
        b = ins + find + erase
    return {"bytes": int(b), "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The outputs from the inputs alone: a stored key gives its value, any other gives 0."""
    c, dev = case, _dev()
    s = _inputs(c, seed, dev)
    kind = c["kind"]

    def found(q, is_hit, val=_values):
        v = val(c, q)
        return torch.where(is_hit, v, torch.zeros_like(v)), is_hit.to(torch.uint8)

    def ones(n):
        return torch.ones(n, dtype=torch.uint8, device=dev)

    if kind == "upsert":
        vals, hit = found(s["q"], s["is_hit"])
        changed = torch.isin(s["q"], s["k"])
        vals = torch.where(changed & s["is_hit"], _new_values(c, s["q"]), vals)
        return (torch.isin(s["k"], s["old"]).to(torch.uint8), vals, hit, ones(s["fresh"].numel()),
                ones(s["old"].numel()), c["keys"])
    out = found(s["q"], s["is_hit"])
    if kind == "load":
        if "zq" in s:
            out = out + found(s["zq"], torch.ones_like(s["zq"], dtype=torch.bool))
        return out + (c["keys"],)
    if kind == "churn":
        return out + (ones(c["n"]), c["keys"])
    if kind == "resize":
        return out + out + (c["keys"],)
    if kind == "host":
        vals, hit = (x.cpu().numpy() for x in out)
        return vals.view(np.uint32), hit, np.ones(c["n"], dtype=np.uint8)
    if kind == "serve":
        return out + (ones(s["q"].numel()),)
    return out
