"""The one-block scan and the radix sort's smaller tiles at the sizes where
they change: scans through the seed expansion (a max-scan of its size), sorts
through the query lists (two sorts of their entries)."""
import ctypes

import numpy as np
import pytest

import gz_native as gz
import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1, 2, 1023, 1024, 1025, 2048, 2049, 16383, 16384, 16385, 50001])
def test_scan_sizes(size):
    rng = np.random.default_rng(size)
    L = gz.lib()
    starts = np.flatnonzero(np.r_[True, rng.random(size - 1) < 0.3]).astype(np.uint32)
    runs = starts.size
    table = rng.integers(0, 10**6, (2, 900)).astype(np.uint32)
    ids = rng.integers(0, 900, runs).astype(np.uint32)
    print("scan: items", size, "runs", runs, flush=True)
    keep = [gz.DeviceBuffer.from_array(x) for x in table]
    h = ctypes.c_void_p()
    gz.check(L.gz_ungapped_extender_create(ctypes.byref(h)))
    gz.check(L.gz_ungapped_extender_set_query_seed_data_list(h, keep[0].ptr, keep[1].ptr))
    tb = L.gz_ungapped_extender_query_seeds_temp_bytes(size)
    temp, tmp = gz.DeviceBuffer(tb), gz.DeviceBuffer(size * 4)
    d_ids, d_starts = gz.DeviceBuffer(runs * 4), gz.DeviceBuffer(runs * 4)
    qid, qpos = gz.DeviceBuffer(size * 4), gz.DeviceBuffer(size * 4)
    s = gz.Stream()
    gz.check(L.gz_ungapped_extender_set_query_seeds(
        h, runs, size, gz.ptr(ids), gz.ptr(starts), tb, temp.ptr, d_ids.ptr, d_starts.ptr,
        qid.ptr, qpos.ptr, tmp.ptr, s.handle))
    s.sync()
    L.gz_ungapped_extender_destroy(h)
    run = np.searchsorted(starts, np.arange(size), side="right") - 1
    assert np.array_equal(qid.to_array(np.uint32, size), table[0][ids[run]])
    assert np.array_equal(qpos.to_array(np.uint32, size), table[1][ids[run]])


# entries from a few to past the last change of the tile size (131,072)
@pytest.mark.parametrize("reads", [1, 12, 200, 330, 390, 600, 780, 1100])
def test_lists_by_entries(reads):
    gz.check(gz.lib().gz_set_device(0))
    qd, dd = synthetic.translated_workload(60 + reads, 300, reads)
    q, db = gz.Queries(*qd, translated=True), gz.Database(*dd)
    host = gz.query_lists(q, db, on_device=False)
    dev = gz.query_lists(q, db, on_device=True)
    print("lists: reads", reads, "entries", len(host["entry_queries"]), flush=True)
    for k in ("hash", "entry_offsets", "entry_positions", "entry_queries", "entry_checks"):
        assert np.array_equal(host[k], dev[k]), k
