"""The gapped extension with one wave per job and the row in registers
(wave_dp.h) against the CPU oracle, and against the lane-per-job form that
calls of more than 131,072 jobs (of queries past 62 residues) take.  All outputs are whole numbers and are
compared exactly."""
import ctypes

import numpy as np
import pytest

import gz_native as gz
import oracle_py
from helpers import DELIM, concat, mutate, random_protein

pytestmark = pytest.mark.gpu
WAVE_JOBS = 131072


def pairs(rng, lengths, identity, indel):
    """Related pairs (query, database) with a seed on a shared diagonal."""
    qs, ds = [], []
    for n in lengths:
        a = random_protein(rng, int(n), 0.02)
        b = mutate(rng, a, rng.uniform(*identity), indel)
        qs.append(a)
        ds.append(b if len(b) else random_protein(rng, 3))
    q, qo = concat(qs)
    d, do = concat(ds)
    k = np.array([rng.integers(0, min(qo[i + 1] - qo[i], do[i + 1] - do[i]) - 1 or 1)
                  for i in range(len(lengths))])
    return q, d, (qo[:-1] + k).astype(np.uint32), (do[:-1] + k).astype(np.uint32)


def extend(q, d, qpos, dpos, reverse, cutoff, gap_open=11, gap_ext=1, order=None, told=4000):
    L, n = gz.lib(), qpos.size
    m, nl = gz.blosum62()
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    dm = gz.DeviceBuffer.from_array(m)
    h = ctypes.c_void_p()
    gz.check(L.gz_gapped_extender_create(ctypes.byref(h)))
    gz.check(L.gz_gapped_extender_set_queries(h, DELIM, pq.ptr))
    gz.check(L.gz_gapped_extender_set_database(h, pd.ptr))
    gz.check(L.gz_gapped_extender_set_score_parameters(h, dm.ptr, nl, gap_open, gap_ext, cutoff))
    gz.check(L.gz_gapped_extender_set_max_sequence_length(h, told))
    s = gz.Stream()
    dq, dd = gz.DeviceBuffer.from_array(qpos), gz.DeviceBuffer.from_array(dpos)
    ds, dc = gz.DeviceBuffer(4 * n), gz.DeviceBuffer(4 * n)
    if order is None:
        gz.check(L.gz_gapped_extender_extend_one_side_score_only_cells_async(
            h, n, int(reverse), dq.ptr, dd.ptr, ds.ptr, dc.ptr, s.handle))
    else:
        do = gz.DeviceBuffer.from_array(order.astype(np.uint32))
        gz.check(L.gz_gapped_extender_extend_one_side_score_only_ordered_async(
            h, n, int(reverse), do.ptr, dq.ptr, dd.ptr, ds.ptr, dc.ptr, s.handle))
    s.sync()
    f = (ctypes.c_uint32 * 1)()
    gz.check(L.gz_gapped_extender_failures(h, f))
    assert f[0] == 0
    out = [ds.to_array(np.int32, n), dq.to_array(np.uint32, n), dd.to_array(np.uint32, n),
           dc.to_array(np.uint32, n)]
    L.gz_gapped_extender_destroy(h)
    return out


def oracle(q, d, qpos, dpos, reverse, cutoff, gap_open, gap_ext):
    m, nl = gz.blosum62()
    out = np.zeros((qpos.size, 3), np.int64)
    for i, (a, b) in enumerate(zip(qpos, dpos)):
        s, p0, p1, _, _ = oracle_py.gapped_one_side("oracle", q, int(a), q.size, d, int(b), DELIM,
                                                    reverse, m, nl, gap_open, gap_ext, cutoff)
        out[i] = s, int(a) + p0, int(b) + p1
    return out


# windows of 64 and of 128 columns and bands past both; sides that end inside
# the first window, at its edge and past it; the parameters' ends
@pytest.mark.parametrize("cutoff,gap_open,gap_ext,lengths", [
    (26, 11, 1, (1, 2, 3, 11, 12, 13, 23, 24, 25, 47, 48, 49, 50, 62, 63, 64, 65, 66, 67)),
    (26, 11, 1, (127, 128, 129, 300, 1500)),
    (0, 11, 1, (5, 70)), (11, 11, 1, (5, 70)), (12, 11, 1, (30, 90)),
    (52, 11, 1, (40, 63, 64, 65, 127, 128, 129, 700)),
    (120, 11, 1, (60, 130, 900)), (120, 0, 1, (40, 400)), (60, 0, 3, (40, 400)),
    (35, 8, 0, (40, 63, 64, 200))])
@pytest.mark.parametrize("reverse", [False, True])
def test_rows_vs_oracle(cutoff, gap_open, gap_ext, lengths, reverse):
    rng = np.random.default_rng(cutoff * 7 + gap_open + len(lengths) + int(reverse))
    print("rows: cutoff", cutoff, "gaps", gap_open, gap_ext, "reverse", reverse, flush=True)
    q, d, qpos, dpos = pairs(rng, np.repeat(lengths, 12), (0.25, 1.0), 0.05)
    if reverse:
        qpos, dpos = qpos - 1, dpos - 1
    s, qe, de, _ = extend(q, d, qpos, dpos, reverse, cutoff, gap_open, gap_ext)
    want = oracle(q, d, qpos, dpos, reverse, cutoff, gap_open, gap_ext)
    got = np.stack([s, qe, de], 1).astype(np.int64)
    bad = np.nonzero((got != want).any(1))[0]
    assert bad.size == 0, (bad[:5], got[bad[:5]], want[bad[:5]])


@pytest.mark.parametrize("cutoff", [26, 52])
@pytest.mark.parametrize("reverse", [False, True])
def test_rows_equal_lanes(cutoff, reverse):
    """WAVE_JOBS + 37 jobs in one call (a lane per job, wide bands to the
    waves) and the same jobs in calls that take a wave per job, in order and
    through a permutation: scores, positions and DP cells."""
    rng = np.random.default_rng(cutoff + int(reverse))
    q, d, qpos, dpos = pairs(rng, rng.integers(20, 220, 1500), (0.3, 1.0), 0.04)
    if reverse:
        qpos, dpos = qpos - 1, dpos - 1
    n = WAVE_JOBS + 37
    pick = rng.integers(0, qpos.size, n)
    print("rows and lanes: cutoff", cutoff, "jobs", n, flush=True)
    one = extend(q, d, qpos, dpos, reverse, cutoff)
    many = extend(q, d, qpos[pick], dpos[pick], reverse, cutoff)
    turned = extend(q, d, qpos, dpos, reverse, cutoff, order=rng.permutation(qpos.size))
    for a, b, c in zip(one, many, turned):
        assert np.array_equal(a[pick], b)
        assert np.array_equal(a, c)


# the two- and the four-column kernel and what decides between them and the
# lanes: sides around 126 and 254 residues and past 2,046 told, bands that
# start past 64 columns, lose a row to a gap and outgrow 128 and 256
@pytest.mark.parametrize("cutoff,gap_open,gap_ext", [
    (26, 11, 1), (26, 5, 1), (42, 11, 1), (43, 11, 1), (73, 11, 1), (74, 11, 1), (90, 11, 1),
    (99, 11, 1), (105, 11, 1), (120, 11, 1), (120, 0, 1), (26, 11, 0), (60, 0, 0), (60, 2, 3),
    (120, 500, 12)])
@pytest.mark.parametrize("told,lengths", [
    (62, (1, 40, 60, 61, 62)), (126, (63, 64, 100, 124, 125, 126)),
    (2046, (126, 127, 128, 129, 253, 254, 255, 256, 257, 700)), (2047, (300, 2047))])
@pytest.mark.parametrize("reverse", [False, True])
def test_windows_vs_oracle(told, lengths, cutoff, gap_open, gap_ext, reverse):
    rng = np.random.default_rng(told + 7 * cutoff + gap_open)
    print("windows: told", told, "cutoff", cutoff, "gaps", gap_open, gap_ext, reverse, flush=True)
    q, d, qpos, dpos = pairs(rng, np.repeat(lengths, 8), (0.25, 1.0), 0.05)
    if reverse:
        qpos, dpos = qpos - 1, dpos - 1
    s, qe, de, _ = extend(q, d, qpos, dpos, reverse, cutoff, gap_open, gap_ext, told=told)
    want = oracle(q, d, qpos, dpos, reverse, cutoff, gap_open, gap_ext)
    got = np.stack([s, qe, de], 1).astype(np.int64)
    bad = np.nonzero((got != want).any(1))[0]
    assert bad.size == 0, (bad[:5], got[bad[:5]], want[bad[:5]])
