"""The distance and ungapped extender kernels where their word-wise forms can
go wrong: window lengths around the twelve codes of a word, calls around the
size from which a lane takes several pairs, cutoffs around the range of the
pair walk, other delimiters and matrices.  Compared exactly with the oracle."""
import ctypes

import numpy as np
import pytest

import gz_native as gz
import oracle_py
from helpers import DELIM, related_pair_set

pytestmark = pytest.mark.gpu
SEVERAL_PAIRS = 2048 * 256 * 2


def distances(q, d, qc, dc, length, rmap):
    L, n = gz.lib(), qc.size
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    d_map = gz.DeviceBuffer.from_array(rmap)
    dq, dd, out = gz.DeviceBuffer.from_array(qc), gz.DeviceBuffer.from_array(dc), gz.DeviceBuffer(n)
    h = ctypes.c_void_p()
    gz.check(L.gz_distance_calculator_create(ctypes.byref(h)))
    gz.check(L.gz_distance_calculator_set_queries(h, pq.ptr))
    gz.check(L.gz_distance_calculator_set_database(h, pd.ptr))
    gz.check(L.gz_distance_calculator_set_reduced_code_map(h, d_map.ptr))
    gz.check(L.gz_distance_calculator_set_subsequence_length(h, length))
    s = gz.Stream()
    gz.check(L.gz_distance_calculator_calculate_distances_async(
        h, n, None, None, None, dq.ptr, dd.ptr, out.ptr, s.handle))
    s.sync()
    L.gz_distance_calculator_destroy(h)
    return out.to_array(np.int8, n)


def centres(rng, n):
    q, qo, d, do, _, _ = related_pair_set(rng, 200, min_len=5, max_len=120)
    # any place, delimiters inside the window too, and both ends
    qc = rng.integers(0, len(q), n).astype(np.uint32)
    dc = rng.integers(0, len(d), n).astype(np.uint32)
    qc[:4], dc[:4] = (0, len(q) - 1, 0, len(q) - 1), (0, len(d) - 1, len(d) - 1, 0)
    return q, d, qc, dc


@pytest.mark.parametrize("length", [0, 1, 5, 6, 7, 10, 11, 12, 13, 24, 25, 36])
def test_distance_lengths(length):
    rng = np.random.default_rng(length)
    q, d, qc, dc = centres(rng, 3001)
    rmap, _ = gz.reduced_map()
    print("distances: length", length, flush=True)
    got = distances(q, d, qc, dc, length, rmap)
    pad = np.full(48, DELIM, np.uint8)
    qp, dp = np.concatenate([pad, q, pad]), np.concatenate([pad, d, pad])
    cls = np.concatenate([rmap[:25], 100 + np.arange(25, 32)]).astype(np.int64)
    k = np.arange(length)[None, :] - length // 2 + 48
    want = (cls[qp[qc[:, None] + k]] != cls[dp[dc[:, None] + k]]).sum(1)
    assert np.array_equal(got, want.astype(np.int8))


@pytest.mark.parametrize("n", [1, 255, 257, SEVERAL_PAIRS, SEVERAL_PAIRS + 1, 3 * 524288 + 77])
def test_distance_call_sizes(n):
    rng = np.random.default_rng(n)
    q, d, qc, dc = centres(rng, 4099)
    rmap, _ = gz.reduced_map()
    print("distances: pairs", n, flush=True)
    one = distances(q, d, qc, dc, 10, rmap)
    pick = rng.integers(0, qc.size, n)
    assert np.array_equal(distances(q, d, qc[pick], dc[pick], 10, rmap), one[pick])


@pytest.mark.parametrize("low,high", [(-3, 2), (1, 12), (100, 128), (127, 131), (129, 400)])
@pytest.mark.parametrize("delim,scale", [(DELIM, 1), (7, 1), (DELIM, 11)])
def test_ungapped_cutoffs(low, high, delim, scale):
    """Cutoffs in and past the pair walk's range; a delimiter that is a letter
    of the matrix; scores up to the ends of a byte."""
    rng = np.random.default_rng(low + 5 * delim + scale)
    q, _, d, _, qpos, dpos = related_pair_set(rng, 1500, min_len=5, max_len=300)
    # delim in the frame, as the sequences of a program with that delimiter
    if delim != DELIM:
        for a in (q, d):
            a[a == delim] = 0
            a[a == DELIM] = delim
    m, nl = gz.blosum62()
    m = np.clip(m.astype(np.int64) * scale, -127, 127).astype(np.int32)
    n = qpos.size
    cut = rng.integers(low, high + 1, n).astype(np.int32)
    trig = rng.integers(5, 60 * scale, n).astype(np.int32)
    print("ungapped: cutoffs", low, high, "delimiter", delim, "scale", scale, flush=True)
    L = gz.lib()
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    keep = [gz.DeviceBuffer.from_array(x) for x in
            (cut, trig, m, np.arange(n, dtype=np.uint32), qpos, dpos)]
    out = gz.DeviceBuffer(n)
    h = ctypes.c_void_p()
    gz.check(L.gz_ungapped_extender_create(ctypes.byref(h)))
    gz.check(L.gz_ungapped_extender_set_queries(h, delim, pq.ptr, keep[0].ptr, keep[1].ptr))
    gz.check(L.gz_ungapped_extender_set_database(h, pd.ptr))
    gz.check(L.gz_ungapped_extender_set_score_matrix(h, keep[2].ptr, nl))
    s = gz.Stream()
    gz.check(L.gz_ungapped_extender_extend_with_trigger_async(
        h, n, None, None, None, None, keep[3].ptr, keep[4].ptr, keep[5].ptr, out.ptr, None,
        s.handle))
    s.sync()
    L.gz_ungapped_extender_destroy(h)
    O = oracle_py.oracle()
    want = np.array([O.gzo_ungapped_with_trigger(gz.ptr(q), int(a), gz.ptr(d), int(b), delim,
                                                 gz.ptr(m), nl, int(c), int(t)) > int(t)
                     for a, b, c, t in zip(qpos, dpos, cut, trig)], np.int8)
    assert np.array_equal(out.to_array(np.int8, n), want)
