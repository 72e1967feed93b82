"""Bulk calls that sort their batch by table region first (partition.hpp):
sizes around the passes' edges (one and two sorting passes, ragged tiles, a
last region of few windows), duplicate-heavy and skewed batches (segments
that overflow), invalid keys, limited probing, batches on top of stored keys,
and tables that more than one stream modifies."""
import math

import numpy as np
import pytest
import torch

from datagen import dev_empty, dtype, from_dev, to_dev, tomb, uniform_values, unique_keys

pytestmark = pytest.mark.gpu

S_NONE, S_PLE, S_INVALID_KEY, S_DUP, S_NOT_FOUND = 0, 2, 8, 16, 32
S_OUT_OF_MEMORY, S_MAX_VALUES = 1 << 7, 1 << 11
SENTINEL = 0x5A5A5A5A


def _batch(n, bits, shape, seed):
    """n keys: distinct, or with the duplicates `shape` names."""
    rng = np.random.default_rng(seed)
    keys = unique_keys(n, bits, seed)
    if shape == "repeats":          # every eighth key twice
        keys[: n // 8] = keys[n - n // 8:]
        rng.shuffle(keys)
    elif shape == "hot":            # two keys take half of the batch
        keys[::3] = keys[1]
        keys[1::7] = keys[2]
    elif shape == "few":            # about fifty copies of each key: region segments overflow
        keys = keys[rng.integers(0, max(1, n // 50), n)]
    elif shape == "invalid":
        keys[::997] = 0
        keys[3::1009] = tomb(bits)
    return np.ascontiguousarray(keys)


def _value_of(keys, bits):
    x = keys.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(0x7F4A7C15)
    return (x >> np.uint64(64 - bits)).astype(dtype(bits)) if bits == 32 else x


def _valid(keys, bits):
    return (keys != 0) & (keys != tomb(bits))


def _status_counts(keys, st, bits):
    """Per distinct valid key: how many `none` among its statuses."""
    ok = _valid(keys, bits)
    uniq, inv = np.unique(keys[ok], return_inverse=True)
    return np.bincount(inv, weights=(st[ok] == S_NONE), minlength=len(uniq))


@pytest.mark.parametrize("kb,vb,cg,n,load,shape", [
    (64, 64, 8, 1 << 20, 0.9, "distinct"),
    (64, 64, 8, (1 << 21) + 4095, 0.93, "repeats"),
    (64, 64, 8, 5_000_001, 0.9, "distinct"),      # more than 1024 regions: two passes
    (64, 64, 8, 5_000_001, 0.9, "hot"),
    (64, 64, 8, 4_500_000, 0.9, "few"),
    (64, 64, 16, 2_000_003, 0.8, "invalid"), (64, 64, 4, 1_500_001, 0.9, "repeats"),
    (32, 32, 16, 12_000_001, 0.9, "distinct"), (32, 32, 16, (1 << 21) - 1, 0.95, "few"),
    (32, 32, 8, 1 << 20, 0.8, "hot"), (32, 32, 8, 9_000_007, 0.9, "repeats"), (32, 32, 4, 1 << 20, 0.9, "invalid"),
    (32, 64, 8, 1_234_567, 0.9, "repeats"), (64, 32, 8, 6_400_000, 0.9, "hot"),
])
@pytest.mark.parametrize("statuses", [False, True])
def test_insert(cuda, kb, vb, cg, n, load, shape, statuses):
    from warpcore_amd.tables import SingleValueHashTable
    keys = _batch(n, kb, shape, seed=n + cg)
    vals = _value_of(keys, vb)
    t = SingleValueHashTable(math.ceil(n / load), kb, vb, cg_size=cg)
    st = dev_empty(n, 32, 0x77)
    t.insert(to_dev(keys), to_dev(vals), status_out=st if statuses else None)
    valid = _valid(keys, kb)
    uniq = np.unique(keys[valid])
    assert t.size() == len(uniq)
    word = (S_DUP if len(uniq) < valid.sum() else 0) | (S_INVALID_KEY if not valid.all() else 0)
    assert int(t.pop_status()) == word
    if statuses:
        got = from_dev(st, np.uint32)
        assert (got[~valid] == S_INVALID_KEY).all()
        assert set(np.unique(got[valid])) <= {S_NONE, S_DUP}
        assert (_status_counts(keys, got, kb) == 1).all()
    out, found = dev_empty(n, vb, SENTINEL), dev_empty(n, 32, 0x77)
    t.retrieve(to_dev(keys), out, status_out=found)
    found = from_dev(found, np.uint32)
    assert (found[valid] == S_NONE).all() and (found[~valid] == S_INVALID_KEY).all()
    np.testing.assert_array_equal(from_dev(out, dtype(vb))[valid], vals[valid])
    absent = unique_keys(100_000, kb, seed=3, exclude=uniq)
    out = dev_empty(len(absent), vb, SENTINEL)
    t.retrieve(to_dev(absent), out, status_out=st[: len(absent)])
    assert (from_dev(st[: len(absent)], np.uint32) == S_NOT_FOUND).all()
    assert (from_dev(out, dtype(vb)) == SENTINEL).all()


@pytest.mark.parametrize("kb,cg", [(64, 8), (32, 16)])
def test_insert_limited_probing(cuda, kb, cg):
    """One window per key: keys past a full first window report
    probing_length_exceeded, and exactly the others are stored."""
    from warpcore_amd.tables import SingleValueHashTable
    n = 3_000_017
    keys = unique_keys(n, kb, seed=5)
    t = SingleValueHashTable(math.ceil(n / 0.95), kb, kb, cg_size=cg)
    st = dev_empty(n, 32, 0x77)
    t.insert(to_dev(keys), to_dev(keys), status_out=st, probing_length=cg)
    st = from_dev(st, np.uint32)
    assert set(np.unique(st)) == {S_NONE, S_PLE}
    assert int(t.pop_status()) == S_PLE
    assert t.size() == (st == S_NONE).sum()
    out, found = dev_empty(n, kb, SENTINEL), dev_empty(n, 32, 0x77)
    t.retrieve(to_dev(keys), out, status_out=found, probing_length=cg)
    found = from_dev(found, np.uint32)
    np.testing.assert_array_equal(found == S_NONE, st == S_NONE)


@pytest.mark.parametrize("kb,vb,cg", [(64, 64, 8), (32, 32, 8)])
def test_insert_on_stored_keys(cuda, kb, vb, cg):
    """Half of the keys stored one small batch at a time before (another
    kernel, other slot orders), some erased; then all of them at once."""
    from warpcore_amd.tables import SingleValueHashTable
    n = 1_300_003
    keys = unique_keys(n, kb, seed=9)
    old = uniform_values(n, vb, seed=10)
    t = SingleValueHashTable(math.ceil(n / 0.8), kb, vb, cg_size=cg)
    half = n // 2
    for lo in range(0, half, 100_000):
        hi = min(lo + 100_000, half)
        t.insert(to_dev(keys[lo:hi]), to_dev(old[lo:hi]))
    t.erase(to_dev(keys[:1000]))
    st = dev_empty(n, 32, 0x77)
    t.insert(to_dev(keys), to_dev(_value_of(keys, vb)), status_out=st)
    st = from_dev(st, np.uint32)
    assert (st[:1000] == S_NONE).all() and (st[1000:half] == S_DUP).all() and (st[half:] == S_NONE).all()
    assert t.size() == n
    out = dev_empty(n, vb, SENTINEL)
    t.retrieve(to_dev(keys), out)
    np.testing.assert_array_equal(from_dev(out, dtype(vb)), _value_of(keys, vb))


def _sorted(insert):
    """Whether insert() sorts its batch by region: what it leaves in the
    library's workspace after a trim."""
    from warpcore_amd.tables import trim_workspace, workspace_bytes
    trim_workspace()
    insert()
    return workspace_bytes() > 0


def test_inserts_from_two_streams(cuda):
    """Batches large enough for the region passes on two streams, without
    synchronization: the first one on `a` is sorted, the one on `b` waits for
    it and takes the general kernels, as everything does until init()."""
    from warpcore_amd.tables import SingleValueHashTable
    n = 2_000_000   # 0.41 of the slots
    keys = unique_keys(2 * n, 64, seed=21)
    vals = _value_of(keys, 64)
    kd, vd = to_dev(keys), to_dev(vals)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    t = SingleValueHashTable(math.ceil(2 * n / 0.9), 64, 64)
    assert t.capacity() * 3 // 8 < n

    def part(i, s):
        t.insert(kd[i * n:(i + 1) * n], vd[i * n:(i + 1) * n], stream=s)

    torch.cuda.synchronize()
    for round_ in range(3):
        t.init(stream=a)
        part(0, a)
        part(1, b)
        torch.cuda.synchronize()
        assert t.size() == 2 * n
        out = torch.zeros_like(vd)
        t.retrieve(kd, out, stream=a)
        torch.cuda.synchronize()
        assert torch.equal(out, vd)
    t.init(stream=a)
    assert _sorted(lambda: part(0, a))
    assert not _sorted(lambda: part(1, b))
    assert not _sorted(lambda: part(0, a))   # the table has seen two streams
    t.init(stream=a)
    assert _sorted(lambda: part(0, a)) and _sorted(lambda: part(1, a))
    torch.cuda.synchronize()
    assert t.size() == 2 * n


def test_inserts_before_under_and_after_capture(cuda):
    """A captured insert's graph may be replayed at any time: from the capture
    on the table's inserts are the general ones; the graph is replayed between
    and after them."""
    from warpcore_amd.tables import SingleValueHashTable
    n = 2_000_000
    keys = unique_keys(2 * n, 64, seed=22)
    kd, vd = to_dev(keys), to_dev(_value_of(keys, 64))
    t = SingleValueHashTable(math.ceil(2 * n / 0.9), 64, 64)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    assert _sorted(lambda: t.insert(kd[:n], vd[:n], stream=s))
    g = torch.cuda.CUDAGraph()
    other = torch.zeros_like(vd[:n])
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        t.insert(kd[n:], other, stream=s)
    out = torch.zeros_like(vd)
    for replay in range(3):
        other.copy_(vd[n:] + replay)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert t.size() == 2 * n
        t.retrieve(kd, out)
        assert torch.equal(out[:n], vd[:n]) and torch.equal(out[n:], other)
        assert not _sorted(lambda: t.insert(kd[:n], vd[:n], stream=s))
        t.init(stream=s)
        torch.cuda.synchronize()
        assert not _sorted(lambda: t.insert(kd[:n], vd[:n], stream=s))


@pytest.mark.parametrize("before", [False, True])
def test_insert_beside_a_capture_of_another_stream(cuda, before):
    """A bulk insert whose workspace is allocated while another stream is
    captured in the global mode: the insert runs, the capture stays valid;
    also where the captured stream ran the region insert `before` whose end
    the table and the workspace wait for."""
    from warpcore_amd.tables import BloomFilter, SingleValueHashTable, trim_workspace
    n = 3_000_001
    keys = unique_keys(n, 64, seed=23)
    kd, vd = to_dev(keys), to_dev(_value_of(keys, 64))
    t, bf = SingleValueHashTable(math.ceil(n / 0.85), 64, 64), BloomFilter(1 << 26, 4, 64)
    x = torch.zeros(1024, device="cuda")
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    trim_workspace()
    torch.cuda.synchronize()
    if before:
        t.insert(kd, vd, stream=b)
    with torch.cuda.graph(g, stream=b, capture_error_mode="global"):
        x.add_(1)
        t.insert(kd, vd, stream=a)
        bf.insert(kd, stream=a)
        x.add_(2)
    out, flags = torch.zeros_like(vd), torch.zeros(n, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    t.retrieve(kd, out)
    bf.retrieve(kd, flags)
    assert torch.equal(out, vd) and bool((flags == 1).all()) and t.size() == n
    for replay in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert bool((x == 3 * (replay + 1)).all())


def test_workspace_is_given_back(cuda):
    """Kept between inserts and reused, given back by a trim, by the last
    table's end, and where a table's own allocation needs the memory; refused
    where it would take more than half of what is free."""
    import gc
    from warpcore_amd.tables import HashSet, SingleValueHashTable, trim_workspace, workspace_bytes
    gc.collect()
    trim_workspace()
    assert workspace_bytes() == 0
    n = 20_000_003
    keys = unique_keys(n, 64, seed=27)
    kd = to_dev(keys)
    t = SingleValueHashTable(math.ceil(n / 0.85), 64, 64)
    small = SingleValueHashTable(1 << 22, 64, 64)
    small.insert(kd[:3_000_000], kd[:3_000_000])
    first = workspace_bytes()
    assert 0 < first < 1 << 30
    t.insert(kd, kd)
    held = workspace_bytes()
    assert held > first
    small.init()
    small.insert(kd[:3_000_000], kd[:3_000_000])
    t.init()
    t.insert(kd, kd)
    assert workspace_bytes() == held
    # a card as good as full: the next table gets the workspace's memory
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    want = (held - first) // 2
    hog = []
    while len(hog) < 8 and torch.cuda.mem_get_info()[0] >= want:
        hog.append(torch.empty(torch.cuda.mem_get_info()[0] - want // 2, dtype=torch.uint8, device="cuda"))
    assert torch.cuda.mem_get_info()[0] < want
    late = HashSet(want // 8, 64)
    assert int(late.peek_status()) == S_NONE and workspace_bytes() == 0
    # too little left for a workspace: the insert runs without
    out = torch.zeros_like(kd[:1 << 20])
    small.init()
    small.insert(kd[:3_000_000], kd[:3_000_000])
    small.retrieve(kd[:1 << 20], out)
    assert small.size() == 3_000_000 and torch.equal(out, kd[:1 << 20])
    del hog, late
    torch.cuda.empty_cache()
    small.init()
    small.insert(kd[:3_000_000], kd[:3_000_000])
    assert workspace_bytes() == first and trim_workspace() == first and workspace_bytes() == 0
    t.init()
    t.insert(kd, kd)
    t.retrieve(kd[:1 << 20], out)
    assert t.size() == n and torch.equal(out, kd[:1 << 20])


def test_other_inserts_without_a_workspace(cuda, oracle):
    """Sets, counters, filters and bucket lists where too little memory is free
    for a workspace: the general kernels."""
    from warpcore_amd.tables import (BloomFilter, BucketListHashTable, CountingHashTable, HashSet, trim_workspace,
                                     workspace_bytes)
    n = 5_000_001
    keys = unique_keys(n, 64, seed=29)
    kd = to_dev(keys)
    h, c = HashSet(math.ceil(n / 0.9), 64), CountingHashTable(math.ceil(n / 0.9), 64)
    bf, bl = BloomFilter(1 << 27, 4, 64), BucketListHashTable(math.ceil(n / 2 / 0.9), 2 * n, 64, 64)
    six = kd[: n // 6].repeat(6)
    flags, counts = torch.zeros(n, dtype=torch.uint8, device="cuda"), torch.zeros(n, dtype=torch.int64, device="cuda")
    c.insert(kd)   # its own combining buffers
    c.init()
    trim_workspace()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hog = []
    while len(hog) < 8 and torch.cuda.mem_get_info()[0] >= 64 << 20:
        hog.append(torch.empty(torch.cuda.mem_get_info()[0] - (40 << 20), dtype=torch.uint8, device="cuda"))
    free = torch.cuda.mem_get_info()[0]
    h.insert(kd)
    c.insert(kd)
    bf.insert(kd)
    bl.insert(six, six)
    held = workspace_bytes()
    del hog
    torch.cuda.empty_cache()
    assert free < 64 << 20 and held == 0
    h.contains(kd, flags)
    assert h.size() == n and bool((flags == 1).all())
    c.retrieve(kd, counts)
    assert c.size() == n and bool((counts == 1).all())
    ob = oracle.Bloom(1 << 27, 4, 64, 64, 1, bf.seed())
    ob.insert(keys)
    np.testing.assert_array_equal(from_dev(bf.words(), np.uint64), ob.words())
    assert bl.num_keys() == n // 6 and bl.num_values() == n // 6 * 6


def test_batches_of_more_than_one_chunk(cuda):
    """More keys than one run of the passes takes (2^28), into each kind."""
    from warpcore_amd import _capi
    from warpcore_amd.tables import BloomFilter, BucketListHashTable, HashSet, SingleValueHashTable
    n = (1 << 28) + (1 << 27) + 3
    keys = torch.empty(n, dtype=torch.int32, device="cuda")
    assert _capi.lib().wc_gen_unique_u32(keys.data_ptr(), n, 0x9000, None) == 0
    h = HashSet(math.ceil(n / 0.9), 32)
    assert _sorted(lambda: h.insert(keys))
    flags = torch.zeros(n, dtype=torch.uint8, device="cuda")
    h.contains(keys, flags)
    assert h.size() == n and int((flags != 1).sum()) == 0
    del h
    print("[chunks] set done", flush=True)
    t = SingleValueHashTable(math.ceil(n / 0.9), 32, 32, cg_size=16)
    st = torch.full((n,), 0x77, dtype=torch.int32, device="cuda")
    assert _sorted(lambda: t.insert(keys, keys, status_out=st))
    out = torch.zeros_like(keys)
    t.retrieve(keys, out)
    assert t.size() == n and torch.equal(out, keys) and int((st != S_NONE).sum()) == 0
    del t, st
    print("[chunks] table done", flush=True)
    one, pieces = BloomFilter(1 << 30, 3, 32), BloomFilter(1 << 30, 3, 32)
    assert _sorted(lambda: one.insert(keys))
    for lo in range(0, n, 1 << 25):
        pieces.insert(keys[lo:lo + (1 << 25)])
    assert torch.equal(one.words(), pieces.words())
    del one, pieces
    print("[chunks] filter done", flush=True)
    d = 1 << 24
    owner = keys[:d].repeat(n // d + 1)[:n]
    bl = BucketListHashTable(math.ceil(d / 0.9), 2 * n, 32, 32)
    assert _sorted(lambda: bl.insert(owner, owner))
    begin, end = (torch.zeros(d, dtype=torch.int64, device="cuda") for _ in range(2))
    assert bl.retrieve(keys[:d], begin, end, out) == n
    count = torch.full((d,), n // d, dtype=torch.int64, device="cuda")
    count[: n % d] += 1
    assert torch.equal(end - begin, count) and torch.equal(out, torch.repeat_interleave(keys[:d], count))


def _streams_side_by_side():
    """Two streams whose kernels do run beside each other (streams share a few
    hardware queues)."""
    x = torch.zeros(1024, device="cuda")
    for _ in range(16):
        a, b = torch.cuda.Stream(), torch.cuda.Stream()
        after = torch.cuda.Event()
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)
            after.record(a)
        with torch.cuda.stream(b):
            x.add_(1)
        b.synchronize()
        beside = not after.query()
        torch.cuda.synchronize()
        if beside:
            return a, b
    pytest.skip("no two streams run beside each other")


def test_insert_does_not_wait_for_another_stream(cuda):
    """Stream a's insert is queued behind a long kernel; an insert into
    another table on stream b ends before that kernel does."""
    from warpcore_amd.tables import SingleValueHashTable
    n = 3_000_001
    keys = unique_keys(n, 64, seed=25)
    kd, vd = to_dev(keys), to_dev(_value_of(keys, 64))
    ta, tb = (SingleValueHashTable(math.ceil(n / 0.85), 64, 64) for _ in range(2))
    a, b = _streams_side_by_side()
    after = torch.cuda.Event()
    ta.insert(kd, vd, stream=b)   # a workspace that both could use
    ta.init(stream=b)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(1_000_000_000)   # some tenths of a second
        after.record(a)
    ta.insert(kd, vd, stream=a)
    tb.insert(kd, vd, stream=b)
    b.synchronize()
    assert not after.query()   # the kernel on a still runs
    torch.cuda.synchronize()
    out = torch.zeros_like(vd)
    for t in (ta, tb):
        out.zero_()
        t.retrieve(kd, out)
        assert torch.equal(out, vd) and t.size() == n


@pytest.mark.parametrize("kb,n,load,shape", [
    (32, 1 << 20, 0.9, "distinct"), (32, 16_000_003, 0.9, "repeats"),   # one pass and two
    (32, 3_000_001, 0.93, "hot"), (32, 16_000_003, 0.9, "few"),
    (64, 1_500_001, 0.9, "invalid"), (64, 8_000_009, 0.9, "repeats"),
])
@pytest.mark.parametrize("statuses", [False, True])
def test_set_insert(cuda, kb, n, load, shape, statuses):
    from warpcore_amd.tables import HashSet
    keys = _batch(n, kb, shape, seed=n)
    h = HashSet(math.ceil(n / load), kb)
    st = dev_empty(n, 32, 0x77)
    h.insert(to_dev(keys), status_out=st if statuses else None)
    valid = _valid(keys, kb)
    uniq = np.unique(keys[valid])
    assert h.size() == len(uniq)
    word = (S_DUP if len(uniq) < valid.sum() else 0) | (S_INVALID_KEY if not valid.all() else 0)
    assert int(h.pop_status()) == word
    if statuses:
        got = from_dev(st, np.uint32)
        assert (got[~valid] == S_INVALID_KEY).all()
        assert (_status_counts(keys, got, kb) == 1).all()
    flags = torch.zeros(n, dtype=torch.uint8, device="cuda")
    h.contains(to_dev(keys), flags)
    assert bool((flags.cpu().numpy()[valid] == 1).all())
    absent = unique_keys(100_000, kb, seed=3, exclude=uniq)
    flags.fill_(7)
    h.contains(to_dev(absent), flags[: len(absent)])
    assert int(flags[: len(absent)].sum()) == 0


@pytest.mark.parametrize("kb,n,distinct,skew", [
    (64, 1 << 22, 1 << 20, 0.0), (64, 9_000_001, 3_700_000, 0.0), (64, 9_000_001, 3_700_000, 1.1),
    (32, 6_000_003, 1_000_003, 0.7),
])
@pytest.mark.parametrize("statuses", [False, True])
def test_counting_insert(cuda, kb, n, distinct, skew, statuses):
    """Counts of two calls on top of each other, the second on keys half new."""
    from warpcore_amd.tables import CountingHashTable
    rng = np.random.default_rng(n)
    uniq = unique_keys(distinct, kb, seed=n)
    t = CountingHashTable(math.ceil(distinct / 0.85), kb)
    total = np.zeros(distinct, np.int64)
    for call in range(2):
        hi = distinct // 2 if call == 0 else distinct
        w = np.arange(1, hi + 1, dtype=np.float64) ** -skew
        pick = np.searchsorted(np.cumsum(w / w.sum()), rng.random(n)).clip(max=hi - 1)
        before = total > 0
        total += np.bincount(pick, minlength=distinct)
        st = dev_empty(n, 32, 0x77)
        t.insert(to_dev(uniq[pick]), status_out=st if statuses else None)
        if statuses:
            got = from_dev(st, np.uint32)
            assert set(np.unique(got)) <= {S_NONE, S_DUP}
            none = np.bincount(pick, weights=(got == S_NONE), minlength=distinct)
            np.testing.assert_array_equal(none, (total > 0) & ~before)
    assert int(t.pop_status()) == S_DUP
    assert t.size() == (total > 0).sum()
    out, found = dev_empty(distinct, 64, 0), dev_empty(distinct, 32, 0x77)
    t.retrieve(to_dev(uniq), out, status_out=found)
    np.testing.assert_array_equal(from_dev(out, np.int64) * (total > 0), total)
    np.testing.assert_array_equal(from_dev(found, np.uint32) == S_NONE, total > 0)


@pytest.mark.parametrize("kb", [32, 64])
@pytest.mark.parametrize("n", [(1 << 22) - 1, 1 << 22, (1 << 23) + 8191])
@pytest.mark.parametrize("shape", ["one", "few", "distinct"])
def test_counting_large_pass(cuda, kb, n, shape):
    """Combining without statuses at the size where a pass takes the larger
    tile: one key only, a few, as many as occurrences; invalid keys between."""
    from warpcore_amd.tables import CountingHashTable
    distinct = {"one": 1, "few": 3000, "distinct": n}[shape]
    uniq = unique_keys(distinct, kb, seed=n + 1)
    pick = np.random.default_rng(n).permutation(n) % distinct
    keys = uniq[pick]
    bad = np.array([5, n // 2, n - 1])
    keys[bad] = [0, np.iinfo(keys.dtype).max, 0]
    t = CountingHashTable(math.ceil(distinct / 0.9) + 64, kb)
    t.insert(to_dev(keys))
    total = np.bincount(np.delete(pick, bad), minlength=distinct)
    out = dev_empty(distinct, 64, 0)
    t.retrieve(to_dev(uniq), out)
    np.testing.assert_array_equal(from_dev(out, np.int64) * (total > 0), total)
    assert t.size() == (total > 0).sum()


def test_counting_with_maximum(cuda):
    """A maximum count: the general insert, which stops there."""
    from warpcore_amd.tables import CountingHashTable
    uniq = unique_keys(1 << 20, 64, seed=4)
    keys = np.tile(uniq, 5)
    t = CountingHashTable(1 << 21, 64, max_count=3)
    t.insert(to_dev(keys))
    out = dev_empty(len(uniq), 64, 0)
    t.retrieve(to_dev(uniq), out)
    assert (from_dev(out, np.uint64) == 3).all()


@pytest.mark.parametrize("kb,sb,num_bits,k,n,shape", [
    (64, 64, 1 << 26, 8, 1 << 20, "distinct"),
    (64, 64, (1 << 30) - 4096 * 64 + 64, 5, 3_000_017, "distinct"),   # 2048 regions, a short last one
    (64, 32, 40_000_003, 4, 2_000_001, "hot"), (32, 64, 9_999_999, 7, 1_500_000, "few"),
    (32, 32, (1 << 16) + 1, 3, (1 << 20) + 1, "distinct"),            # regions of one word
])
def test_bloom_insert(cuda, oracle, kb, sb, num_bits, k, n, shape):
    from warpcore_amd.tables import BloomFilter
    keys = _batch(n, kb, shape, seed=n)
    bf = BloomFilter(num_bits, k, kb, slot_bits=sb)
    ob = oracle.Bloom(num_bits, k, kb, sb, 1, bf.seed())
    for part in (keys[: n // 2], keys):   # the second call on top of the first
        bf.insert(to_dev(part))
        ob.insert(part)
        np.testing.assert_array_equal(from_dev(bf.words(), dtype(sb)), ob.words())


_WARM = [6000] * 40 + [150_000]   # pairs of the keys that overflow segments


def _sample(n):
    """Positions whose keys decide whether a batch is taken for skewed."""
    return np.arange(4096) * (n // 4096)


def _pair_batch(n, bits, distinct, shape, seed):
    """n pairs over `distinct` keys with distinct values, some keys invalid."""
    rng = np.random.default_rng(seed)
    uniq = unique_keys(distinct, bits, seed=seed + 1)
    if shape == "heavy":     # a share of the batch on few keys: the general insert takes it
        w = np.arange(1, distinct + 1, dtype=np.float64) ** -1.2
        pick = np.searchsorted(np.cumsum(w / w.sum()), rng.random(n)).clip(max=distinct - 1)
    else:
        pick = rng.integers(0, distinct, n)
        if shape == "warm":  # keys of some thousand pairs, none of them sampled (part_begin)
            at = rng.permutation(np.setdiff1d(np.arange(n), _sample(n)))
            pick[at[: sum(_WARM)]] = np.repeat(np.arange(len(_WARM)), _WARM)
    keys = uniq[pick]
    if shape == "invalid":
        keys[::9973] = 0
        keys[1::9967] = tomb(bits)
    return np.ascontiguousarray(keys), np.arange(1, n + 1).astype(dtype(bits)), uniq


def _values_by_key(t, uniq, bits, total):
    """Every key's values, sorted, from one retrieve."""
    begin, end = dev_empty(len(uniq), 64, 0), dev_empty(len(uniq), 64, 0)
    out = dev_empty(total + 1, bits, 0)
    assert t.retrieve(to_dev(uniq), begin, end, out[:total]) == total
    b, e, v = from_dev(begin, np.int64), from_dev(end, np.int64), from_dev(out, dtype(bits))[:total]
    assert b[0] == 0 and e[-1] == total and (b[1:] == e[:-1]).all()
    owner = np.repeat(np.arange(len(uniq)), e - b)
    return owner, v[np.lexsort((v, owner))]


def _expected_by_key(keys, values, uniq):
    order = np.argsort(uniq, kind="stable")
    at = np.searchsorted(uniq[order], keys)
    pos = order[at.clip(max=len(uniq) - 1)]
    ok = uniq[pos] == keys
    owner, v = pos[ok], values[ok]
    by = np.lexsort((v, owner))
    return owner[by], v[by]


@pytest.mark.parametrize("bits,n,distinct,shape", [
    (32, 1 << 20, 1 << 17, "even"), (32, (1 << 20) + 1, 1 << 20, "invalid"), (32, 3_000_017, 300_000, "warm"),
    (32, 1_500_000, 50_000, "heavy"), (64, (1 << 20) + 4097, 90_001, "invalid"), (64, (1 << 23) + 5, 3_000_000, "even"),
])
def test_pairs_insert(cuda, bits, n, distinct, shape):
    """Two calls, the second on top of the first's keys."""
    from warpcore_amd.tables import BucketListHashTable
    keys, values, uniq = _pair_batch(n, bits, distinct, shape, seed=n)
    t = BucketListHashTable(math.ceil(distinct / 0.9) + 64, 4 * n + 4096, bits, bits)
    ok = _valid(keys, bits)
    stored = len(np.unique(keys[ok]))
    for call in range(2):
        t.insert(to_dev(keys), to_dev(values))
        status = int(t.pop_status())
        assert status & ~(S_DUP | S_INVALID_KEY) == 0
        assert bool(status & S_INVALID_KEY) == (not ok.all())
        assert t.num_keys() == stored
        want = _expected_by_key(np.tile(keys[ok], call + 1), np.tile(values[ok], call + 1), uniq)
        got = _values_by_key(t, uniq, bits, (call + 1) * int(ok.sum()))
        t.pop_status()   # key_not_found of the keys that the batch does not hold
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])


@pytest.mark.parametrize("cg,n,distinct,passes", [(4, 1_600_007, 160_000, 1), (8, 3_000_017, 300_000, 2),
                                                  (8, 12_000_001, 1_200_000, 2)])
def test_pairs_insert_with_overflowing_segments(cuda, cg, n, distinct, passes):
    """Keys of 6,000 pairs, more than a region's share, and one of 150,000, more
    than a bucket's: their records take the pair-by-pair rest (several lanes
    append to one key at once), the others the groups."""
    import ctypes
    from pathlib import Path
    from warpcore_amd.tables import BucketListHashTable
    keys, values, uniq = _pair_batch(n, 32, distinct, "warm", seed=n)
    assert np.unique(keys[_sample(n)], return_counts=True)[1].max() < 4   # not taken for skewed
    t = BucketListHashTable(math.ceil(distinct / 0.9), 5 * n, 32, 32, cg_size=cg)
    plan = (ctypes.c_uint64 * 4)()
    ctypes.CDLL(str(Path(__file__).parent / "device_api" / "libwc_device_api.so")).wcx_group_plan(
        ctypes.c_uint(cg), ctypes.c_uint64(n), ctypes.c_uint64(t.key_capacity()), plan)
    cap1, cap2, buckets, two = list(plan)
    assert two == passes - 1 and n >= t.key_capacity()
    # an eighth of a key's pairs on each XCD, beside the mean of the others
    assert 150_000 // 8 + n // 8 // buckets > cap1
    if two:
        assert 6000 > cap2
    assert _sorted(lambda: t.insert(to_dev(keys), to_dev(values)))
    assert int(t.pop_status()) == S_DUP
    got, want = _values_by_key(t, uniq, 32, n), _expected_by_key(keys, values, uniq)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])


@pytest.mark.parametrize("min_size,grow,max_size", [(1, 1.0, 1), (3, 1.1, 1023), (8, 2.0, 64), (1, 1.001, 1023)])
def test_pairs_insert_bucket_shapes(cuda, min_size, grow, max_size):
    from warpcore_amd.tables import BucketListHashTable
    n, distinct = 1_300_000, 60_000
    keys, values, uniq = _pair_batch(n, 32, distinct, "even", seed=7)
    t = BucketListHashTable(70_000, 6 * n, 32, 32, grow_factor=grow, min_bucket_size=min_size, max_bucket_size=max_size)
    for call in range(2):
        t.insert(to_dev(keys), to_dev(values))
    assert int(t.pop_status()) == S_DUP
    want = _expected_by_key(np.tile(keys, 2), np.tile(values, 2), uniq)
    got = _values_by_key(t, uniq, 32, 2 * n)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])


def test_pairs_insert_limits(cuda):
    """A per-key maximum, and a pool too small for the batch."""
    from warpcore_amd.tables import BucketListHashTable
    n, distinct = 1_200_000, 60_000
    keys, values, uniq = _pair_batch(n, 32, distinct, "even", seed=9)
    have = np.bincount(np.searchsorted(np.sort(uniq), keys), minlength=distinct)
    t = BucketListHashTable(70_000, 4 * n, 32, 32, max_values_per_key=10)
    t.insert(to_dev(keys), to_dev(values))
    assert int(t.pop_status()) == S_DUP | S_MAX_VALUES
    owner, v = _values_by_key(t, np.sort(uniq), 32, int(np.minimum(have, 10).sum()))
    np.testing.assert_array_equal(np.bincount(owner, minlength=distinct), np.minimum(have, 10))
    assert len(np.unique(v)) == len(v) and (np.sort(uniq)[owner] == keys[v.astype(np.int64) - 1]).all()
    small = BucketListHashTable(70_000, n // 2, 32, 32)
    small.insert(to_dev(keys), to_dev(values))
    assert int(small.pop_status()) & (S_OUT_OF_MEMORY | S_DUP) == S_OUT_OF_MEMORY | S_DUP
    total = small.num_values()
    assert n // 8 < total <= n // 2
    owner, v = _values_by_key(small, uniq, 32, total)
    assert len(np.unique(v)) == total and (uniq[owner] == keys[v.astype(np.int64) - 1]).all()


@pytest.mark.parametrize("distinct", [1 << 18, 1 << 20])
def test_pairs_insert_tight_pool(cuda, distinct):
    """Eight values per key in buckets of 1, 2, 3 and 4 (13 cells) and a pool
    of just so many cells and, per arena, the 4 that a bucket of 5 cells may
    leave: everything is stored."""
    from warpcore_amd.tables import BucketListHashTable
    n = 8 * distinct
    keys = np.tile(unique_keys(distinct, 32, seed=distinct), 8)
    np.random.default_rng(3).shuffle(keys)
    kd, vd = to_dev(keys), torch.arange(n, dtype=torch.int32, device="cuda")
    arenas = 1
    while arenas < 256 and 13 * distinct // (2 * arenas) >= 1 << 16:
        arenas *= 2
    t = BucketListHashTable(math.ceil(distinct / 0.9), 13 * distinct + 4 * arenas, 32, 32, grow_factor=1.1,
                            min_bucket_size=1)
    t.insert(kd, vd)
    assert int(t.pop_status()) == S_DUP
    assert t.num_keys() == distinct and t.num_values() == n
