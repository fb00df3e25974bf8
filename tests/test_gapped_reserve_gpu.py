"""gz_gapped_extender_reserve: calls of up to the reserved jobs allocate
nothing, whichever form (a wave or a lane per job) the settings of the call
choose and however much shorter its queries are told, and give what a new
handle gives."""
import ctypes

import numpy as np
import pytest

import gz_native as gz
from helpers import DELIM, related_pair_set

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("told", [500, 65534])
def test_reserve_holds_for_later_settings(told):
    L, n = gz.lib(), 20000
    rng = np.random.default_rng(told)
    q, _, d, _, qpos, dpos = related_pair_set(rng, 400, min_len=20, max_len=480)
    qpos, dpos = np.resize(qpos, n).astype(np.uint32), np.resize(dpos, n).astype(np.uint32)
    m, nl = gz.blosum62()
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    dm = gz.DeviceBuffer.from_array(m)
    s = gz.Stream()
    dq, dd, ds = (gz.DeviceBuffer(4 * n) for _ in range(3))

    def handle(told):
        h = ctypes.c_void_p()
        gz.check(L.gz_gapped_extender_create(ctypes.byref(h)))
        gz.check(L.gz_gapped_extender_set_queries(h, DELIM, pq.ptr))
        gz.check(L.gz_gapped_extender_set_database(h, pd.ptr))
        gz.check(L.gz_gapped_extender_set_max_sequence_length(h, told))
        return h

    def run(h, jobs, cutoff, gaps):
        gz.check(L.gz_gapped_extender_set_score_parameters(h, dm.ptr, nl, *gaps, cutoff))
        gz.check(L.gz_memcpy_async(dq.ptr, gz.ptr(qpos), 4 * n, s.handle))
        gz.check(L.gz_memcpy_async(dd.ptr, gz.ptr(dpos), 4 * n, s.handle))
        gz.check(L.gz_gapped_extender_extend_one_side_score_only_async(
            h, jobs, 0, None, None, None, dq.ptr, dd.ptr, ds.ptr, s.handle))
        s.sync()
        f = (ctypes.c_uint32 * 1)()
        gz.check(L.gz_gapped_extender_failures(h, f))
        assert f[0] == 0

    def outputs(jobs):
        return [x.to_array(np.uint32, jobs) for x in (ds, dq, dd)]

    h = handle(told)
    gz.check(L.gz_gapped_extender_set_score_parameters(h, dm.ptr, nl, 11, 1, 26))
    gz.check(L.gz_gapped_extender_reserve(h, n, s.handle))
    s.sync()
    for shorter in (told, 500):
        gz.check(L.gz_gapped_extender_set_max_sequence_length(h, shorter))
        for jobs, cutoff, gaps in ((n, 26, (11, 1)), (n, 130, (11, 1)), (n, 26, (600, 1)),
                                   (n // 2 + 1, 1100, (11, 1))):
            print("reserved: told", told, shorter, "jobs", jobs, cutoff, gaps, flush=True)
            one = handle(500)  # first, so that the kernels have run before
            run(one, jobs, cutoff, gaps)
            want = outputs(jobs)
            L.gz_gapped_extender_destroy(one)
            before = free_bytes()
            run(h, jobs, cutoff, gaps)
            assert free_bytes() == before
            for a, b in zip(outputs(jobs), want):
                assert np.array_equal(a, b)
    L.gz_gapped_extender_destroy(h)
