"""Performance cases of the hash tables, over the sizes a user runs them at.

A case is one whole piece of work of a program that uses the tables through
``warpcore_amd.tables``: building a table and probing it (a hash join), a
small lookup against a resident table, building, erasing and probing,
counting, set membership, Bloom filtering, multi-value builds and gathers,
many small tables at once, and a burst of served requests. ``listed()`` names
the fixed cases, ``draw()`` gives more of the same ranges.

Every output is an integer that the inputs determine (stored values, counts,
flags, statuses, offsets), so every case is compared exactly. Keys are
distinct scrambled counters, as the benchmark's are; where the order in which
equal keys arrive is free (the values of one key of a multi-value table), the
values of a key are equal, so that the output does not depend on that order.
"""
from __future__ import annotations

import math

import torch

from warpcore_amd.tables import (BloomFilter, BucketListHashTable, CountingHashTable, HashSet, MultiValueHashTable,
                                 Server, SingleValueHashTable, TableBatch)

_INT = {32: torch.int32, 64: torch.int64}
_MASK64 = (1 << 64) - 1


# ------------------------------------------------------------------ inputs --
def _signed(x: int, bits: int) -> int:
    x &= (1 << bits) - 1
    return x - (1 << bits) if x >> (bits - 1) else x


def _fmix64_int(x: int) -> int:
    x &= _MASK64
    x ^= x >> 33
    x = x * 0xFF51AFD7ED558CCD & _MASK64
    x ^= x >> 33
    x = x * 0xC4CEB9FE1A85EC53 & _MASK64
    return x ^ (x >> 33)


def _shift_right(x, s: int):
    """Logical shift of int64 bit patterns."""
    return (x >> s) & ((1 << (64 - s)) - 1)


def _scramble64(x):
    """A bijection of 64-bit words (in place on an int64 tensor)."""
    for mul in (0xFF51AFD7ED558CCD, 0xC4CEB9FE1A85EC53):
        x ^= _shift_right(x, 33)
        x *= _signed(mul, 64)
    x ^= _shift_right(x, 33)
    return x


def _scramble32(x):
    """A bijection of 32-bit words held in an int64 tensor (in place)."""
    m = 0xFFFFFFFF
    x ^= x >> 16
    for mul, s in ((0x85EBCA6B, 13), (0xC2B2AE35, 16)):
        x *= mul
        x &= m
        x ^= x >> s
    return x


def _keys(count: int, bits: int, seed: int, first: int = 0):
    """Keys number first .. first + count of the seed's sequence of distinct
    keys, none of them 0 or ~0 (EMPTY and TOMBSTONE)."""
    out = torch.empty(count, dtype=_INT[bits], device="cuda")
    salt = _fmix64_int(seed * 2 + 1)
    step = 1 << 26
    for lo in range(0, count, step):
        x = torch.arange(first + lo, first + min(lo + step, count), dtype=torch.int64, device="cuda")
        if bits == 64:
            x += (salt >> 2) + 1
            x = _scramble64(x)
            x[(x == 0) | (x == -1)] = _signed(_fmix64_int((salt >> 2) - 7), 64)
        else:
            x += 16
            x *= salt & 0xFFFF | 1
            x &= 0xFFFFFFFF
            x = _scramble32(x)
            # the first 16 numbers are never used otherwise: two of them stand in for 0 and ~0
            for bad, number in ((0, 5), (0xFFFFFFFF, 9)):
                spare = torch.tensor([number * (salt & 0xFFFF | 1) & 0xFFFFFFFF], device="cuda")
                x[x == bad] = _scramble32(spare)[0]
        out[lo: lo + x.numel()] = x.to(_INT[bits])
    return out


def _generator(seed: int):
    g = torch.Generator(device="cuda")
    g.manual_seed(_fmix64_int(seed) >> 1)
    return g


def _words(count: int, bits: int, seed: int):
    return torch.randint(-(1 << (bits - 1)), (1 << (bits - 1)) - 1, (count,), dtype=_INT[bits], device="cuda",
                         generator=_generator(seed + 77))


def _value_of(keys, bits: int):
    """A value that the key determines."""
    x = keys.to(torch.int64)
    x = x * 0x9E3779B1 + 0x7F4A7C15
    return (x ^ _shift_right(x, 29)).to(_INT[bits])


def _queries(stored, count: int, hit: float, bits: int, seed: int):
    """`count` lookups, a share `hit` of them stored keys (each drawn at
    random), the others absent, in random order."""
    g = _generator(seed + 13)
    absent = _keys(count, bits, seed, first=stored.numel())
    step = 1 << 26
    for lo in range(0, count, step):
        n = min(step, count - lo)
        pick = torch.randint(0, stored.numel(), (n,), device="cuda", generator=g)
        is_hit = torch.rand(n, device="cuda", generator=g) < hit
        part = absent[lo: lo + n]
        part.copy_(torch.where(is_hit, stored[pick], part))
    return absent


def _power_law(count: int, distinct: int, s: float, seed: int):
    """`count` ranks below `distinct`, the share of rank r falling as r**-s."""
    g = _generator(seed + 31)
    out = torch.empty(count, dtype=torch.int32, device="cuda")
    step = 1 << 26
    a = 1.0 - s
    for lo in range(0, count, step):
        u = torch.rand(min(step, count - lo), device="cuda", dtype=torch.float64, generator=g)
        x = torch.pow(u * ((distinct + 1.0) ** a - 1.0) + 1.0, 1.0 / a)
        out[lo: lo + u.numel()] = (x.long() - 1).clamp_(0, distinct - 1).to(torch.int32)
    return out


def _pairs(count: int, mean: float, bits: int, seed: int):
    """`count` (key, value) pairs in random order over about count / mean
    distinct keys whose multiplicities are geometric; and those keys."""
    distinct = max(1, int(count / mean))
    g = _generator(seed + 57)
    weight = -torch.log1p(-torch.rand(distinct, device="cuda", dtype=torch.float64, generator=g))
    cumulative = torch.cumsum(weight, 0)
    cumulative /= cumulative[-1].clone()
    keys = _keys(distinct, bits, seed)
    out = torch.empty(count, dtype=_INT[bits], device="cuda")
    step = 1 << 25
    for lo in range(0, count, step):
        u = torch.rand(min(step, count - lo), device="cuda", dtype=torch.float64, generator=g)
        out[lo: lo + u.numel()] = keys[torch.searchsorted(cumulative, u).clamp_(max=distinct - 1)]
    return out, _value_of(out, bits), keys


def _status(count: int, wanted: bool):
    return torch.zeros(count, dtype=torch.int32, device="cuda") if wanted else None


def _given(**outputs):
    return {k: v for k, v in outputs.items() if v is not None}


# ------------------------------------------------------- the kinds of work --
class _Join:
    """Build a table of distinct keys, then probe it (a hash join): init,
    insert, retrieve."""

    @staticmethod
    def prepare(c, seed):
        kb, vb, n, m = c["key_bits"], c["value_bits"], c["keys"], c["queries"]
        keys = _keys(n, kb, seed)
        s = {"keys": keys, "values": _words(n, vb, seed), "queries": _queries(keys, m, c["hit"], kb, seed),
             "out": torch.zeros(m, dtype=_INT[vb], device="cuda"),
             "inserted": _status(n, c["statuses"]), "found": _status(m, c["statuses"]),
             "table": SingleValueHashTable(math.ceil(n / c["load"]), kb, vb, cg_size=c["cg"])}
        return s

    @staticmethod
    def run(s):
        t = s["table"]
        t.init()
        t.insert(s["keys"], s["values"], status_out=s["inserted"])
        t.retrieve(s["queries"], s["out"], status_out=s["found"])
        return _given(out=s["out"], inserted=s["inserted"], found=s["found"])

    @staticmethod
    def bytes(c):
        kb, vb, n, m = c["key_bits"] // 8, c["value_bits"] // 8, c["keys"], c["queries"]
        slot = max(8, 16 if kb + vb > 8 else 8)
        st = 4 * (n + m) if c["statuses"] else 0
        return n * (kb + vb) + slot * n / c["load"] + m * (kb + slot + vb) + st


class _Lookup:
    """Lookups against a table that stays resident."""

    @staticmethod
    def prepare(c, seed):
        kb, vb, n, m = c["key_bits"], c["value_bits"], c["keys"], c["queries"]
        keys = _keys(n, kb, seed)
        t = SingleValueHashTable(math.ceil(n / c["load"]), kb, vb, cg_size=c["cg"])
        t.insert(keys, _words(n, vb, seed))
        return {"table": t, "queries": _queries(keys, m, c["hit"], kb, seed),
                "out": torch.zeros(m, dtype=_INT[vb], device="cuda"), "found": _status(m, c["statuses"])}

    @staticmethod
    def run(s):
        s["table"].retrieve(s["queries"], s["out"], status_out=s["found"])
        return _given(out=s["out"], found=s["found"])

    @staticmethod
    def bytes(c):
        kb, vb, m = c["key_bits"] // 8, c["value_bits"] // 8, c["queries"]
        return m * (kb + 2 * vb + kb + (4 if c["statuses"] else 0))


class _Churn:
    """Build, erase a quarter of the keys, probe for all of them."""

    @staticmethod
    def prepare(c, seed):
        kb, vb, n = c["key_bits"], c["value_bits"], c["keys"]
        keys = _keys(n, kb, seed)
        return {"keys": keys, "values": _words(n, vb, seed), "gone": keys[: max(1, n // 4)].clone(),
                "queries": _queries(keys, n, 1.0, kb, seed), "out": torch.zeros(n, dtype=_INT[vb], device="cuda"),
                "erased": _status(max(1, n // 4), True), "found": _status(n, True),
                "table": SingleValueHashTable(math.ceil(n / c["load"]), kb, vb, cg_size=c["cg"])}

    @staticmethod
    def run(s):
        t = s["table"]
        t.init()
        t.insert(s["keys"], s["values"])
        t.erase(s["gone"], status_out=s["erased"])
        t.retrieve(s["queries"], s["out"], status_out=s["found"])
        return {"out": s["out"], "erased": s["erased"], "found": s["found"]}

    @staticmethod
    def bytes(c):
        kb, vb, n = c["key_bits"] // 8, c["value_bits"] // 8, c["keys"]
        slot = 16 if kb + vb > 8 else 8
        return n * (kb + vb) + slot * n / c["load"] + n // 4 * (2 * kb + 4) + n * (kb + slot + vb + 4)


class _Count:
    """Occurrences of skewed keys, then the counts of all candidate keys."""

    @staticmethod
    def prepare(c, seed):
        n, d, kb = c["occurrences"], c["distinct"], c["key_bits"]
        candidates = _keys(d, kb, seed)
        ranks = _power_law(n, d, c["skew"], seed)
        occurrences = torch.empty(n, dtype=_INT[kb], device="cuda")
        step = 1 << 26
        for lo in range(0, n, step):
            occurrences[lo: lo + step] = candidates[ranks[lo: lo + step].long()]
        return {"keys": occurrences, "candidates": candidates, "found": _status(d, c["statuses"]),
                "counts": torch.zeros(d, dtype=torch.int64, device="cuda"),
                "table": CountingHashTable(math.ceil(d / c["load"]), kb)}

    @staticmethod
    def run(s):
        t = s["table"]
        t.init()
        t.insert(s["keys"])
        t.retrieve(s["candidates"], s["counts"], status_out=s["found"])
        return _given(counts=s["counts"], found=s["found"])

    @staticmethod
    def bytes(c):
        kb, n, d = c["key_bits"] // 8, c["occurrences"], c["distinct"]
        return n * kb + 16 * d / c["load"] + d * (kb + 16 + 8 + (4 if c["statuses"] else 0))


class _Set:
    """Insert keys into a set, then test present and absent keys."""

    @staticmethod
    def prepare(c, seed):
        kb, n, m = c["key_bits"], c["keys"], c["queries"]
        keys = _keys(n, kb, seed)
        return {"keys": keys, "queries": _queries(keys, m, c["hit"], kb, seed),
                "flags": torch.zeros(m, dtype=torch.uint8, device="cuda"), "inserted": _status(n, c["statuses"]),
                "set": HashSet(math.ceil(n / c["load"]), kb)}

    @staticmethod
    def run(s):
        h = s["set"]
        h.init()
        h.insert(s["keys"], status_out=s["inserted"])
        h.contains(s["queries"], s["flags"])
        return _given(flags=s["flags"], inserted=s["inserted"])

    @staticmethod
    def bytes(c):
        kb, n, m = c["key_bits"] // 8, c["keys"], c["queries"]
        return n * (kb + (4 if c["statuses"] else 0)) + kb * n / c["load"] + m * (2 * kb + 1)


class _Bloom:
    """Fill a Bloom filter, then query it."""

    @staticmethod
    def prepare(c, seed):
        kb, n, m = c["key_bits"], c["keys"], c["queries"]
        keys = _keys(n, kb, seed)
        return {"keys": keys, "queries": _queries(keys, m, c["hit"], kb, seed),
                "flags": torch.zeros(m, dtype=torch.uint8, device="cuda"),
                "filter": BloomFilter(c["bits"], c["k"], kb)}

    @staticmethod
    def run(s):
        f = s["filter"]
        f.init()
        f.insert(s["keys"])
        f.retrieve(s["queries"], s["flags"])
        return {"flags": s["flags"]}

    @staticmethod
    def bytes(c):
        kb, n, m = c["key_bits"] // 8, c["keys"], c["queries"]
        return n * kb + c["bits"] / 8 + m * (kb + 8 + 1)


class _Multi:
    """Build a multi-value table of pairs, then gather every key's values."""

    @staticmethod
    def prepare(c, seed):
        kb, n = c["bits"], c["pairs"]
        keys, values, distinct = _pairs(n, c["mean"], kb, seed)
        d = distinct.numel()
        if c["kind"] == "multi":
            t = MultiValueHashTable(math.ceil(n / c["load"]), kb, kb)
        else:
            t = BucketListHashTable(math.ceil(d / c["load"]), math.ceil(n * 2.5) + 4096, kb, kb, grow_factor=1.1,
                                    min_bucket_size=1)
        return {"table": t, "keys": keys, "values": values, "distinct": distinct,
                "begin": torch.zeros(d, dtype=torch.int64, device="cuda"),
                "end": torch.zeros(d, dtype=torch.int64, device="cuda"),
                "out": torch.zeros(n, dtype=_INT[kb], device="cuda")}

    @staticmethod
    def run(s):
        t = s["table"]
        t.init()
        t.insert(s["keys"], s["values"])
        total = t.retrieve(s["distinct"], s["begin"], s["end"], s["out"])
        return {"begin": s["begin"], "end": s["end"], "out": s["out"], "total": total}

    @staticmethod
    def bytes(c):
        b, n = c["bits"] // 8, c["pairs"]
        d = n / c["mean"]
        stored = 2 * b * n / c["load"] if c["kind"] == "multi" else 16 * d / c["load"] + 8 * n
        return n * 2 * b + 2 * stored + d * (b + 16) + n * b


class _Batch:
    """Many small tables filled and probed in one call each."""

    @staticmethod
    def prepare(c, seed):
        import numpy as np
        bits = c["bits"]
        rng = np.random.default_rng(c["tables"])   # the sizes belong to the case, the keys to the seed
        caps = np.exp2(rng.uniform(math.log2(c["smallest"]), math.log2(c["largest"]), c["tables"])).astype(np.uint64)
        count = np.maximum((caps * rng.uniform(0.5, 0.9, c["tables"])).astype(np.uint64), 1)
        offsets = np.concatenate([[0], np.cumsum(count)]).astype(np.int64)
        n = int(offsets[-1])
        keys = _keys(n, bits, seed)
        batch = TableBatch(caps, bits, bits, cg_size=c["cg"])
        # the launch that the tuner of a batch of this kind settles on
        batch.set_launch(8192, 16, 128)
        # lookups of every stored key, table by table, one in eight replaced by an absent key
        queries = keys.clone()
        queries[::8] = _keys((n + 7) // 8, bits, seed, first=n)
        return {"batch": batch, "keys": keys, "values": _words(n, bits, seed), "queries": queries,
                "offsets": torch.from_numpy(offsets).to("cuda"), "found": _status(n, c["statuses"]),
                "out": torch.zeros(n, dtype=_INT[bits], device="cuda")}

    @staticmethod
    def run(s):
        b = s["batch"]
        b.init()
        b.insert(s["keys"], s["values"], s["offsets"])
        b.retrieve(s["queries"], s["offsets"], s["out"], status_out=s["found"])
        return _given(out=s["out"], found=s["found"])

    @staticmethod
    def bytes(c):
        b = c["bits"] // 8
        lo, hi = c["smallest"], c["largest"]
        slots = c["tables"] * ((hi - lo) / math.log(hi / lo) if hi > lo else lo)
        n = 0.7 * slots
        return n * 2 * b + slots * 2 * b + n * (b + 2 * b + b + (4 if c["statuses"] else 0))


class _Serve:
    """A burst of requests to the serving loop: lookups and updates of stored
    keys on several resident tables, submitted together, then drained."""

    @staticmethod
    def prepare(c, seed):
        import numpy as np
        rng = np.random.default_rng(c["requests"])   # the requests' shapes belong to the case, the keys to the seed
        bits, tables, per_table = c["bits"], c["tables"], c["keys"]
        server = Server([math.ceil(per_table / 0.5)] * tables, bits, bits)
        stored = [_keys(per_table, bits, seed * 64 + t) for t in range(tables)]
        torch.cuda.synchronize()   # the server runs on a stream of its own
        for t in range(tables):
            values = _value_of(stored[t], bits)
            torch.cuda.synchronize()
            server.wait(server.submit(Server.INSERT, t, stored[t], values_in=values))
        sizes = np.exp2(rng.uniform(math.log2(c["smallest"]), math.log2(c["largest"]), c["requests"])).astype(int)
        sizes = np.minimum(sizes, per_table).tolist()
        out = torch.zeros(sum(sizes), dtype=_INT[bits], device="cuda")
        status = _status(sum(sizes), True)
        requests, lo = [], 0
        for size in sizes:
            t, cut = int(rng.integers(tables)), slice(lo, lo + size)
            lo += size
            if rng.random() < c["updates"]:
                at = int(rng.integers(per_table - size + 1))
                keys = stored[t][at: at + size].clone()
                requests.append((Server.INSERT, t, keys, _value_of(keys, bits), None, status[cut]))
            else:
                keys = _queries(stored[t], size, 0.75, bits, seed * 64 + t)
                requests.append((Server.RETRIEVE, t, keys, None, out[cut], status[cut]))
        return {"server": server, "requests": requests, "out": out, "status": status}

    @staticmethod
    def run(s):
        server = s["server"]
        for op, table, keys, values, out, status in s["requests"]:
            server.submit(op, table, keys, values_in=values, values_out=out, status_out=status)
        server.drain()
        return {"out": s["out"], "status": s["status"]}

    @staticmethod
    def bytes(c):
        lo, hi = c["smallest"], min(c["largest"], c["keys"])
        keys = c["requests"] * ((hi - lo) / math.log(hi / lo) if hi > lo else lo)
        return keys * (c["bits"] // 8 * 4 + 4)


_KINDS = {"join": _Join, "lookup": _Lookup, "churn": _Churn, "count": _Count, "set": _Set, "bloom": _Bloom,
          "multi": _Multi, "buckets": _Multi, "batch": _Batch, "serve": _Serve}


# -------------------------------------------------------------------- cases --
def listed():
    return [
        # the benchmark's headline step: a 4.8 GB table of 64-bit keys at load 0.9, half of the probes absent
        {"name": "join u64 2^28", "kind": "join", "key_bits": 64, "value_bits": 64, "cg": 8, "keys": 1 << 28,
         "queries": 1 << 28, "load": 0.9, "hit": 0.5, "statuses": False},
        # a join side of ordinary size and odd counts, 32-bit keys, statuses asked for, most probes present
        {"name": "join u32 33M statuses", "kind": "join", "key_bits": 32, "value_bits": 32, "cg": 16,
         "keys": 33_333_333, "queries": 50_000_017, "load": 0.8, "hit": 0.8, "statuses": True},
        # the benchmark's small table, resident in the last-level cache
        {"name": "join u32 2^20", "kind": "join", "key_bits": 32, "value_bits": 32, "cg": 8, "keys": 1 << 20,
         "queries": 1 << 21, "load": 0.8, "hit": 0.5, "statuses": False},
        # the smallest call: a request's thousand keys against a resident table
        {"name": "lookup u64 1000", "kind": "lookup", "key_bits": 64, "value_bits": 64, "cg": 8, "keys": 1 << 22,
         "queries": 1000, "load": 0.8, "hit": 0.75, "statuses": True},
        # erasing: build, erase a quarter, probe for everything
        {"name": "churn u64 2^24", "kind": "churn", "key_bits": 64, "value_bits": 64, "cg": 8, "keys": 1 << 24,
         "load": 0.8},
        # counting words or k-mers: skewed occurrences of 2^24 candidate keys
        {"name": "count u64 2^28 skewed", "kind": "count", "key_bits": 64, "occurrences": 1 << 28,
         "distinct": 1 << 24, "skew": 1.1, "load": 0.9, "statuses": False},
        # set membership at the benchmark's size, half of the tests absent
        {"name": "set u32 2^27", "kind": "set", "key_bits": 32, "keys": 1 << 27, "queries": 1 << 27, "load": 0.9,
         "hit": 0.5, "statuses": False},
        # the benchmark's Bloom filter: 8 bits a key, 128 MB
        {"name": "bloom u64 2^27", "kind": "bloom", "key_bits": 64, "keys": 1 << 27, "queries": 1 << 27,
         "bits": 1 << 30, "k": 8, "hit": 0.5},
        # an index of values per key: build and gather, as many slots as pairs
        {"name": "multi u32 2^26", "kind": "multi", "bits": 32, "pairs": 1 << 26, "mean": 8.0, "load": 0.9},
        # the same over growing buckets
        {"name": "buckets u32 2^26", "kind": "buckets", "bits": 32, "pairs": 1 << 26, "mean": 8.0, "load": 0.9},
        # thousands of small tables in one call
        {"name": "batch u32 16384 tables", "kind": "batch", "bits": 32, "tables": 16384, "smallest": 1 << 6,
         "largest": 1 << 16, "cg": 16, "statuses": False},
        # a burst of served requests of 2^8 .. 2^18 keys
        {"name": "serve u64 64 requests", "kind": "serve", "bits": 64, "tables": 8, "keys": 1 << 20, "requests": 64,
         "smallest": 1 << 8, "largest": 1 << 18, "updates": 0.25},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(sorted(_KINDS))
    load = round(rng.uniform(0.5, 0.93), 3)
    hit = round(rng.uniform(0.0, 1.0), 3)
    statuses = rng.random() < 0.35
    if kind == "join":
        kb, vb = rng.choice([(32, 32), (64, 64), (64, 64), (32, 64), (64, 32)])
        n = _log(rng, 1 << 12, 1 << 27)
        return {"kind": kind, "key_bits": kb, "value_bits": vb, "cg": rng.choice([8, 16] if kb == vb == 32 else [8]),
                "keys": n, "queries": max(1, min(1 << 27, int(n * rng.uniform(0.3, 2.5)))), "load": load, "hit": hit,
                "statuses": statuses}
    if kind == "lookup":
        kb, vb = rng.choice([(32, 32), (64, 64), (32, 64), (64, 32)])
        return {"kind": kind, "key_bits": kb, "value_bits": vb, "cg": 8, "keys": _log(rng, 1 << 16, 1 << 25),
                "queries": _log(rng, 1 << 8, 1 << 22), "load": load, "hit": hit, "statuses": statuses}
    if kind == "churn":
        kb, vb = rng.choice([(32, 32), (64, 64)])
        return {"kind": kind, "key_bits": kb, "value_bits": vb, "cg": 8, "keys": _log(rng, 1 << 14, 1 << 26),
                "load": load}
    if kind == "count":
        d = _log(rng, 1 << 12, 1 << 24)
        return {"kind": kind, "key_bits": rng.choice([32, 64]), "occurrences": min(1 << 27, int(d * rng.uniform(2, 40))),
                "distinct": d, "skew": rng.choice([0.4, 0.7, 0.9, 1.1, 1.2]), "load": load, "statuses": statuses}
    if kind == "set":
        n = _log(rng, 1 << 14, 1 << 27)
        return {"kind": kind, "key_bits": rng.choice([32, 64]), "keys": n,
                "queries": max(1, min(1 << 27, int(n * rng.uniform(0.5, 2.0)))), "load": load, "hit": hit,
                "statuses": statuses}
    if kind == "bloom":
        n = _log(rng, 1 << 14, 1 << 27)
        return {"kind": kind, "key_bits": rng.choice([32, 64]), "keys": n,
                "queries": max(1, min(1 << 27, int(n * rng.uniform(0.5, 2.0)))),
                "bits": 64 * max(16, int(n * rng.uniform(6, 16)) // 64), "k": rng.choice([3, 5, 8]), "hit": hit}
    if kind in ("multi", "buckets"):
        return {"kind": kind, "bits": rng.choice([32, 32, 64]), "pairs": _log(rng, 1 << 14, 1 << 26),
                "mean": round(rng.uniform(1.5, 12.0), 2), "load": load}
    if kind == "batch":
        return {"kind": kind, "bits": rng.choice([32, 64]), "tables": _log(rng, 256, 16384), "smallest": 1 << 6,
                "largest": 1 << rng.choice([10, 13, 16]), "cg": 16, "statuses": statuses}
    return {"kind": "serve", "bits": rng.choice([32, 64]), "tables": rng.randint(2, 16),
            "keys": _log(rng, 1 << 16, 1 << 20), "requests": rng.randint(16, 96), "smallest": 1 << 8,
            "largest": 1 << rng.choice([12, 15, 18]), "updates": rng.choice([0.0, 0.25])}


def prepare(case, seed):
    kind = _KINDS[case["kind"]]
    return {"kind": kind, "state": kind.prepare(case, seed)}


def run(state):
    return state["kind"].run(state["state"])


def work(case):
    return {"bytes": float(_KINDS[case["kind"]].bytes(case)), "flops": 0.0}


def tolerance(case):
    return "exact"
