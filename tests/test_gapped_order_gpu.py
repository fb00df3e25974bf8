"""Calls that run a lane per job (more than 65,536 jobs, or 131,072 when the
longest query is told above 62 residues) and bring no order of their own run in
one by query side length (extenders.hip): the results are those of the same
jobs in small calls, at sizes around a block's chunk of 4,096, for sides from none to
past the last bin, with an own delimiter, on every entry point that takes
such calls."""
import ctypes

import numpy as np
import pytest

import gz_native as gz
from helpers import DELIM, concat, mutate, random_protein

pytestmark = pytest.mark.gpu
WAVE_JOBS = 131072  # of queries told longer than 62 residues


def pairs(rng, lengths):
    qs = [random_protein(rng, int(n), 0.02) for n in lengths]
    ds = [mutate(rng, a, rng.uniform(0.3, 1.0), 0.03) for a in qs]
    ds = [b if len(b) > 1 else random_protein(rng, 3) for b in ds]
    q, qo = concat(qs)
    d, do = concat(ds)
    m = np.minimum(np.diff(qo.astype(np.int64)), np.diff(do.astype(np.int64))) - 1
    k = np.array([rng.integers(-1, x + 1) for x in m])  # on the delimiters too
    return q, d, (qo[:-1] + k).astype(np.uint32), (do[:-1] + k).astype(np.uint32)


def extend(q, d, qpos, dpos, reverse, delim, form):
    L, n = gz.lib(), qpos.size
    m, nl = gz.blosum62()
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    dm = gz.DeviceBuffer.from_array(m)
    h = ctypes.c_void_p()
    gz.check(L.gz_gapped_extender_create(ctypes.byref(h)))
    gz.check(L.gz_gapped_extender_set_queries(h, delim, pq.ptr))
    gz.check(L.gz_gapped_extender_set_database(h, pd.ptr))
    gz.check(L.gz_gapped_extender_set_score_parameters(h, dm.ptr, nl, 11, 1, 26))
    gz.check(L.gz_gapped_extender_set_max_sequence_length(h, 400))
    if form == "queue":
        gz.check(L.gz_gapped_extender_set_persistent(h, 1))
    s = gz.Stream()
    dq, dd = gz.DeviceBuffer.from_array(qpos), gz.DeviceBuffer.from_array(dpos)
    ds, dc = gz.DeviceBuffer(4 * n), gz.DeviceBuffer(4 * n)
    call = (L.gz_gapped_extender_extend_one_side_score_only_noalloc_async if form == "noalloc"
            else L.gz_gapped_extender_extend_one_side_score_only_cells_async)
    for _ in range(2):  # the second run finds the first one's counters
        gz.check(L.gz_memcpy_async(dq.ptr, gz.ptr(qpos), 4 * n, s.handle))
        gz.check(L.gz_memcpy_async(dd.ptr, gz.ptr(dpos), 4 * n, s.handle))
        gz.check(call(h, n, int(reverse), dq.ptr, dd.ptr, ds.ptr, dc.ptr, s.handle))
    s.sync()
    f = (ctypes.c_uint32 * 1)()
    gz.check(L.gz_gapped_extender_failures(h, f))
    assert f[0] == 0
    out = [x.to_array(np.uint32, n) for x in (ds, dq, dd, dc)]
    L.gz_gapped_extender_destroy(h)
    return np.stack(out, 1)


@pytest.mark.parametrize("form", ["grid", "queue", "noalloc"])
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("n", [WAVE_JOBS + 1, 33 * 4096, 33 * 4096 + 1, 200003])
def test_order_leaves_results(n, reverse, form):
    rng = np.random.default_rng(n + int(reverse))
    q, d, qpos, dpos = pairs(rng, np.r_[np.arange(1, 140), rng.integers(1, 60, 900)])
    print("order: jobs", n, "reverse", reverse, form, flush=True)
    one = extend(q, d, qpos, dpos, reverse, DELIM, "grid")
    pick = rng.integers(0, qpos.size, n)
    many = extend(q, d, qpos[pick], dpos[pick], reverse, DELIM, form)
    assert np.array_equal(one[pick], many)


def test_order_with_another_delimiter():
    rng = np.random.default_rng(3)
    q, d, qpos, dpos = pairs(rng, rng.integers(1, 90, 700))
    for a in (q, d):  # 31 in the frames, the padding keeps its code
        a[a == DELIM] = 31
    print("order: delimiter 31", flush=True)
    one = extend(q, d, qpos, dpos, False, 31, "grid")
    pick = rng.integers(0, qpos.size, WAVE_JOBS + 999)
    assert np.array_equal(one[pick], extend(q, d, qpos[pick], dpos[pick], False, 31, "grid"))


# past what the order kernels' resident blocks take at once (2,048 chunks of
# 4,096), and past 262,140 chunks, where a grid of one chunk per block ended
@pytest.mark.parametrize("n", [2048 * 4096 + 4097, 262140 * 4096 + 4097])
def test_order_of_large_calls(n):
    L, rng, piece = gz.lib(), np.random.default_rng(7), 1 << 22
    q, d, qpos, dpos = pairs(rng, rng.integers(1, 60, 1000))
    print("order: jobs", n, flush=True)
    m, nl = gz.blosum62()
    one = extend(q, d, qpos, dpos, False, DELIM, "grid")
    pick = rng.integers(0, qpos.size, piece)
    want = one[pick]
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    dm = gz.DeviceBuffer.from_array(m)
    s = gz.Stream()
    arrays = [gz.DeviceBuffer(4 * n) for _ in range(3)]

    def pieces():
        for at in range(0, n, piece):
            yield min(piece, n - at), [ctypes.c_void_p(b.ptr.value + 4 * at) for b in arrays]

    # scores that no job has, so that a job left out is seen
    start = [qpos[pick], dpos[pick], np.full(piece, 0xdeadbeef, np.uint32)]
    for k, at in pieces():
        for a, p in zip(start, at):
            gz.check(L.gz_memcpy_async(p, gz.ptr(a), 4 * k, s.handle))
    s.sync()
    h = ctypes.c_void_p()
    gz.check(L.gz_gapped_extender_create(ctypes.byref(h)))
    gz.check(L.gz_gapped_extender_set_queries(h, DELIM, pq.ptr))
    gz.check(L.gz_gapped_extender_set_database(h, pd.ptr))
    gz.check(L.gz_gapped_extender_set_score_parameters(h, dm.ptr, nl, 11, 1, 26))
    gz.check(L.gz_gapped_extender_set_max_sequence_length(h, 62))
    gz.check(L.gz_gapped_extender_extend_one_side_score_only_async(
        h, n, 0, None, None, None, arrays[0].ptr, arrays[1].ptr, arrays[2].ptr, s.handle))
    s.sync()
    f = (ctypes.c_uint32 * 1)()
    gz.check(L.gz_gapped_extender_failures(h, f))
    L.gz_gapped_extender_destroy(h)
    assert f[0] == 0
    got = [np.empty(piece, np.uint32) for _ in arrays]
    for k, at in pieces():
        for a, p, w in zip(got, at, (1, 2, 0)):
            gz.check(L.gz_memcpy_async(gz.ptr(a), p, 4 * k, s.handle))
            s.sync()
            assert np.array_equal(a[:k], want[:k, w])
