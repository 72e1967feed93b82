"""Device-side tile API (tables passed by value into user kernels), driven
through tests/device_api/libwc_device_api.so: the filtered histogram of
examples/src/advanced_usage_from_device.cu, and insert / retrieve / erase /
multi-value round trips issued from user kernels, checked against the
oracle."""
import ctypes
from pathlib import Path

import numpy as np
import pytest
import torch

from datagen import dev_empty, from_dev, to_dev, unique_keys

pytestmark = pytest.mark.gpu

LIB = Path(__file__).resolve().parent / "device_api" / "libwc_device_api.so"
S_NONE, S_DUP, S_NOT_FOUND = 0, 16, 32


@pytest.fixture(scope="module")
def dlib(cuda):
    if not LIB.exists():
        raise RuntimeError(f"{LIB} is missing: run the build first")
    lib = ctypes.CDLL(str(LIB))
    P, U64, I = ctypes.c_void_p, ctypes.c_uint64, ctypes.c_int
    lib.wcx_filter_and_count_u32.argtypes = [P, U64, U64, P, P, P]
    lib.wcx_svht_create.restype = P
    lib.wcx_svht_create.argtypes = [U64]
    lib.wcx_svht_destroy.argtypes = [P]
    lib.wcx_svht_phase.argtypes = [P, I, P, P, U64, P, P]
    lib.wcx_mvht_roundtrip_u32.argtypes = [P, P, U64, P, U64, U64, P, P, U64, P, P]
    lib.wcx_bucketlist_roundtrip_u32.argtypes = [P, P, U64, P, U64, U64, U64, P, P, U64, P, P]
    return lib


_keep = []


def _p(t):
    """Device pointer of t; t is kept alive until the test module ends (a
    temporary tensor freed before the call could be handed to the next
    allocation)."""
    if t is None:
        return None
    _keep.append(t)
    return ctypes.c_void_p(t.data_ptr())


@pytest.fixture(autouse=True)
def _release():
    yield
    torch.cuda.synchronize()
    _keep.clear()


def test_filtered_histogram_from_device(dlib):
    rng = np.random.default_rng(1)
    uniq = unique_keys(1 << 18, 32, seed=2)
    repeated = unique_keys(1 << 16, 32, seed=3, exclude=uniq)
    keys = np.concatenate([uniq, np.repeat(repeated, 4)])
    rng.shuffle(keys)
    n = len(keys)
    ko, co = dev_empty(n, 32), dev_empty(n, 64)
    num = ctypes.c_uint64(0)
    assert dlib.wcx_filter_and_count_u32(_p(to_dev(keys)), n, 1 << 26, _p(ko), _p(co), ctypes.byref(num)) == 0
    got = dict(zip(from_dev(ko, np.uint32)[: num.value].tolist(), from_dev(co, np.uint64)[: num.value].tolist()))
    # every repeated key is counted 3 times (4 occurrences minus the first),
    # or 4 when the filter gave a false positive on its first occurrence
    rep = set(repeated.tolist())
    exact = sum(1 for k in rep if got.get(k) == 3)
    assert all(got.get(k) in (3, 4) for k in rep)
    extra = [k for k in got if k not in rep]
    # unique keys appear only through false positives (count 1); FPR here is ~1e-6
    assert all(got[k] == 1 for k in extra)
    assert len(extra) + (len(repeated) - exact) <= 8


def test_svht_device_insert_retrieve_erase(dlib, oracle):
    n = 40000
    keys = unique_keys(n, 64, seed=11)
    vals = unique_keys(n, 64, seed=12)
    h = dlib.wcx_svht_create(int(n / 0.8))
    try:
        st = dev_empty(n, 32, 0x77)
        assert dlib.wcx_svht_phase(h, 0, _p(to_dev(keys)), _p(to_dev(vals)), n, None, _p(st)) == 0
        assert np.all(from_dev(st, np.uint32) == S_NONE)
        # re-insert half with new values: duplicates, values overwritten
        vals2 = vals.copy()
        vals2[: n // 2] ^= np.uint64(0xFFFF)
        assert dlib.wcx_svht_phase(h, 0, _p(to_dev(keys[: n // 2])), _p(to_dev(vals2[: n // 2])), n // 2, None,
                                   _p(st)) == 0
        assert np.all(from_dev(st, np.uint32)[: n // 2] == S_DUP)
        absent = unique_keys(1000, 64, seed=13, exclude=keys)
        q = np.concatenate([keys, absent])
        out, qst = dev_empty(len(q), 64, 0x55), dev_empty(len(q), 32)
        assert dlib.wcx_svht_phase(h, 1, _p(to_dev(q)), None, len(q), _p(out), _p(qst)) == 0
        o = oracle.SVHT(int(n / 0.8), 64, 64, cg=8)
        o.insert(keys, vals)
        o.insert(keys[: n // 2], vals2[: n // 2])
        ov, ost = o.retrieve(q)
        np.testing.assert_array_equal(from_dev(qst, np.uint32), ost)
        got = from_dev(out, np.uint64)
        np.testing.assert_array_equal(got[:n], ov[:n])
        # erase a third, then retrieve again
        er = keys[::3]
        est = dev_empty(len(er), 32)
        assert dlib.wcx_svht_phase(h, 2, _p(to_dev(er)), None, len(er), None, _p(est)) == 0
        assert np.all(from_dev(est, np.uint32) == S_NONE)
        o.erase(er)
        out, qst = dev_empty(len(q), 64, 0x55), dev_empty(len(q), 32)
        assert dlib.wcx_svht_phase(h, 1, _p(to_dev(q)), None, len(q), _p(out), _p(qst)) == 0
        ov, ost = o.retrieve(q)
        np.testing.assert_array_equal(from_dev(qst, np.uint32), ost)
        hit = ost == S_NONE
        np.testing.assert_array_equal(from_dev(out, np.uint64)[hit], ov[hit])
    finally:
        dlib.wcx_svht_destroy(h)


def _multi_pairs(num_keys, mean, seed):
    rng = np.random.default_rng(seed)
    keys = unique_keys(num_keys, 32, seed)
    mult = rng.geometric(1.0 / mean, size=num_keys)
    k = np.repeat(keys, mult)
    v = unique_keys(len(k), 32, seed + 1)
    perm = rng.permutation(len(k))
    return keys, mult, k[perm], v[perm]


@pytest.mark.parametrize("kind", ["mvht", "bucketlist"])
def test_multi_value_device_roundtrip(dlib, kind):
    keys, mult, k, v = _multi_pairs(3000, 5.0, seed=21)
    absent = unique_keys(200, 32, seed=23, exclude=keys)
    q = np.concatenate([keys, absent])
    stride = int(mult.max())
    ist = dev_empty(len(k), 32, 0x77)
    vals = dev_empty(len(q) * stride, 32, 0xAB)
    counts, qst = dev_empty(len(q), 64), dev_empty(len(q), 32)
    if kind == "mvht":
        rc = dlib.wcx_mvht_roundtrip_u32(_p(to_dev(k)), _p(to_dev(v)), len(k), _p(to_dev(q)), len(q),
                                         2 * len(k), _p(ist), _p(vals), stride, _p(counts), _p(qst))
    else:
        rc = dlib.wcx_bucketlist_roundtrip_u32(_p(to_dev(k)), _p(to_dev(v)), len(k), _p(to_dev(q)), len(q),
                                               2 * len(keys), 4 * len(k), _p(ist), _p(vals), stride, _p(counts),
                                               _p(qst))
    assert rc == 0
    s = from_dev(ist, np.uint32)
    assert set(np.unique(s)) <= {S_NONE, S_DUP}
    assert np.sum(s == S_NONE) == len(keys)
    c = from_dev(counts, np.uint64)
    np.testing.assert_array_equal(c[: len(keys)], mult.astype(np.uint64))
    assert np.all(c[len(keys):] == 0)
    qs = from_dev(qst, np.uint32)
    assert np.all(qs[: len(keys)] == S_NONE) and np.all(qs[len(keys):] == S_NOT_FOUND)
    got = from_dev(vals, np.uint32).reshape(len(q), stride)
    exp = {}
    for key, val in zip(k.tolist(), v.tolist()):
        exp.setdefault(key, []).append(val)
    for i, key in enumerate(keys.tolist()):
        assert sorted(got[i, : mult[i]].tolist()) == sorted(exp[key])


@pytest.mark.parametrize("max_count,preset", [((1 << 32) - 1, (1 << 32) - 10), (1000, 990), (1000, 1000)])
def test_counting_combined_add_saturates(dlib, max_count, preset):
    """A combined count (one add of all occurrences of a key in a tile) ends
    where single increments would (counting_hash_table.cuh:154-170: each adds
    one while the count is below max_count): min(preset + occurrences,
    max_count), with no index_overflow even where one add would pass 2^32-1."""
    dlib.wcx_counting_u32_saturation.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint32,
                                                 ctypes.c_uint32, ctypes.c_void_p, ctypes.c_void_p,
                                                 ctypes.c_void_p]
    rng = np.random.default_rng(31)
    others = unique_keys(8192, 32, seed=32)
    hot = others[0]
    batch = np.concatenate([np.full(40, hot, np.uint32), others[1:]])
    rng.shuffle(batch)
    batch = np.concatenate([[hot], batch]).astype(np.uint32)   # keys[0] is the preset key
    n = len(batch)
    st, counts = dev_empty(n, 32, 0x77), dev_empty(n, 32, 0x55)
    word = ctypes.c_uint32(0)
    assert dlib.wcx_counting_u32_saturation(_p(to_dev(batch)), n, max_count, preset, _p(st), _p(counts),
                                            ctypes.byref(word)) == 0
    got_s, got_c = from_dev(st, np.uint32), from_dev(counts, np.uint32)
    is_hot = batch == hot
    assert np.all(got_s[is_hot] == S_DUP)            # the key was in the table before the batch
    assert np.all(got_s[~is_hot] == S_NONE)
    assert np.all(got_c[is_hot] == min(preset + int(is_hot.sum()), max_count))
    assert np.all(got_c[~is_hot] == 1)
    assert word.value == S_DUP                        # duplicate_key joined, no index_overflow (64)


def test_inserts_from_threads_on_their_own_null_stream(cuda):
    """The null stream of a translation unit built with
    -fgpu-default-stream=per-thread is another one in every host thread:
    batches large enough for the region passes, none waited for."""
    lib = ctypes.CDLL(str(LIB.with_name("libwc_per_thread.so")))
    lib.wcp_insert_from_threads.restype = ctypes.c_uint64
    lib.wcp_insert_from_threads.argtypes = [ctypes.c_void_p] + [ctypes.c_uint64] * 3 + [ctypes.c_void_p]
    n = 6_000_003   # each half more than 3/8 of the slots
    keys = unique_keys(n, 64, seed=31)
    kd, out = to_dev(keys), dev_empty(n, 64, 0x55)
    torch.cuda.synchronize()
    assert lib.wcp_insert_from_threads(_p(kd), n, 2, int(n / 0.85), _p(out)) == n
    assert torch.equal(out, kd)


@pytest.fixture(scope="module")
def vlib(cuda):
    lib = ctypes.CDLL(str(LIB.with_name("libwc_value_types.so")))
    for f in (lib.wcv_single, lib.wcv_lists):
        f.restype = ctypes.c_int64
        f.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint64]
    return lib


@pytest.mark.parametrize("kind,bits", [(0, 64), (1, 64), (2, 32)])
def test_single_values_of_several_words(vlib, kind, bits):
    """32, 16 and 12 bytes: only the last one's slots fit the region passes' records."""
    n = 3_000_001
    kd = to_dev(unique_keys(n, bits, seed=41 + kind))
    torch.cuda.synchronize()
    assert vlib.wcv_single(kind, _p(kd), n, int(n / 0.9)) == 0


@pytest.mark.parametrize("kind,bits", [(0, 64), (1, 64), (2, 32), (3, 32)])
def test_lists_of_values_of_several_words(vlib, kind, bits):
    n = 1_200_001
    kd = to_dev(unique_keys(n, bits, seed=51 + kind))
    torch.cuda.synchronize()
    assert vlib.wcv_lists(kind, _p(kd), n, int(n / 0.9)) == 0


@pytest.mark.parametrize("which", [0, 1])
def test_status_handler_runs_once_per_key(dlib, which):
    """A batch large enough for the region passes, with duplicates and invalid keys."""
    dlib.wcx_handler_calls.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p]
    n = 3_000_001
    keys = unique_keys(n, 64, seed=61)
    keys[5::5] = keys[1::5]
    keys[::1009] = 0
    kd, calls = to_dev(keys), torch.zeros(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert dlib.wcx_handler_calls(which, _p(kd), n, int(n / 0.9), _p(calls)) == 0
    assert bool((calls == 1).all())


def test_insert_without_host_memory(cuda):
    """Nothing in a bulk insert depends on operator new: no exception leaves
    it, and every key is stored."""
    lib = ctypes.CDLL(str(LIB.with_name("libwc_host_memory.so")))
    lib.wch_insert.restype = ctypes.c_uint64
    lib.wch_insert.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p]
    n = 3_000_001
    kd, out = to_dev(unique_keys(n, 64, seed=71)), dev_empty(n, 64, 0x55)
    torch.cuda.synchronize()
    assert lib.wch_insert(_p(kd), n, int(n / 0.9), _p(out)) == n
    assert torch.equal(out, kd)


@pytest.mark.parametrize("statuses", [0, 1])
def test_lists_with_buckets_larger_than_an_arena(vlib, statuses):
    """Grouped and pair by pair: buckets whose 64-fold size does not fit 32
    bits and of which the pool holds none. Every key is stored, no value is."""
    vlib.wcv_large_buckets.restype = ctypes.c_int64
    vlib.wcv_large_buckets.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_int, ctypes.c_void_p]
    n = 1_300_000   # more pairs than slots
    kd = to_dev(np.tile(unique_keys(20_000, 32, seed=81), n // 20_000))
    word = ctypes.c_uint32(0)
    torch.cuda.synchronize()
    assert vlib.wcv_large_buckets(_p(kd), n, statuses, ctypes.byref(word)) == 0
    assert word.value == S_DUP | 1 << 7   # duplicate_key, out_of_memory


def test_bulk_inserts_beside_a_copy_of_the_table(dlib):
    """A copy handed to a kernel waits for the region insert that still runs,
    and from then on, init() included, bulk inserts run beside anything."""
    P, U64 = ctypes.c_void_p, ctypes.c_uint64
    dlib.wcx_svht_insert.restype = dlib.wcx_svht_init.restype = None
    dlib.wcx_svht_insert.argtypes = [P, P, P, U64, P]
    dlib.wcx_svht_init.argtypes = [P, P]
    dlib.wcx_workspace_bytes.restype = dlib.wcx_workspace_trim.restype = U64
    n, m = 2_000_000, 200_000
    keys = unique_keys(2 * n + m, 64, seed=91)
    kd = to_dev(keys)
    out, st = torch.zeros_like(kd), torch.zeros(len(keys), dtype=torch.int32, device="cuda")
    s = torch.cuda.Stream()   # does not order itself against the null stream, on which the kernels below run
    h = dlib.wcx_svht_create(int(len(keys) / 0.9))
    try:
        torch.cuda.synchronize()
        dlib.wcx_workspace_trim()
        for round_ in range(2):
            dlib.wcx_svht_insert(h, _p(kd), _p(kd), n, P(s.cuda_stream))
            assert (dlib.wcx_workspace_bytes() > 0) == (round_ == 0)
            assert dlib.wcx_svht_phase(h, 0, _p(kd[2 * n:]), _p(kd[2 * n:]), m, None, _p(st)) == 0
            dlib.wcx_workspace_trim()
            dlib.wcx_svht_insert(h, _p(kd[n:]), _p(kd[n:]), n, P(s.cuda_stream))
            assert dlib.wcx_workspace_bytes() == 0
            torch.cuda.synchronize()
            out.zero_()
            torch.cuda.synchronize()
            assert dlib.wcx_svht_phase(h, 1, _p(kd), None, len(keys), _p(out), _p(st)) == 0
            assert torch.equal(out, kd) and int(st.abs().sum()) == 0
            dlib.wcx_svht_init(h, P(s.cuda_stream))
            torch.cuda.synchronize()
    finally:
        dlib.wcx_svht_destroy(h)
