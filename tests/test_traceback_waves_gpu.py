"""The result build with one wave per side (traceback.hip) against the host
result build and the CPU oracle.  All fields are whole numbers and are
compared exactly; a result that reads a byte an earlier extension left must be
flagged as the host flags it."""
import ctypes
import threading

import numpy as np
import pytest

import gz_native as gz
import oracle_py
from helpers import DELIM, concat, mutate, random_protein

pytestmark = pytest.mark.gpu
STALE, OVERFLOW = 1, 2
GAP0, SUB, GAP1 = 0, 1, 2  # the oracle's edits


def jobs_of(rng, lengths, identity, indel, at=None):
    """Related pairs, one job each: the seed at `at` (a share of the shorter
    sequence; None: anywhere) on a shared diagonal."""
    qs, ds = [], []
    for n in lengths:
        a = random_protein(rng, int(n), 0.02)
        b = mutate(rng, a, rng.uniform(*identity), indel)
        qs.append(a)
        ds.append(b if len(b) > 1 else random_protein(rng, 3))
    q, qo = concat(qs)
    d, do = concat(ds)
    jobs = np.zeros((len(qs), 4), np.uint32)
    for i, (a, b) in enumerate(zip(qs, ds)):
        m = min(len(a), len(b))
        k = int(rng.integers(0, m)) if at is None else min(m - 1, int(at * m))
        jobs[i] = qo[i] - 1, len(a) + 2, k + 1, do[i] + k
    return q, d, jobs, int(np.diff(do.astype(np.int64)).max())


def build(q, d, jobs, max_subject, cutoff, gap_open=11, gap_ext=1, max_query=None):
    m, nl = gz.blosum62()
    _, pq = gz.pack_on_device(q)
    _, pd = gz.pack_on_device(d)
    dm = gz.DeviceBuffer.from_array(m)
    jobs = np.ascontiguousarray(jobs)
    out = np.zeros((len(jobs), 10), np.uint32)
    gz.check(gz.lib().gz_build_results(
        pq.ptr, pd.ptr, gz.ptr(jobs), len(jobs),
        int(jobs[:, 1].max()) if max_query is None else max_query, max_subject, dm.ptr, nl,
        gap_open, gap_ext, cutoff, gz.ptr(out), None))
    return out


def on_host(q, d, job, cutoff):
    lead, qlen, hq, hd = (int(x) for x in job)
    qs = np.ascontiguousarray(q[lead:lead + qlen])
    out = np.zeros(10, np.uint32)
    gz.check(gz.lib().gz_build_result_host(gz.ptr(qs), qlen, gz.ptr(d), hq, hd, cutoff,
                                           gz.ptr(out)))
    return out


def by_oracle(q, d, job, cutoff, gap_open, gap_ext):
    """All fields but the flags: scores and ends of the two sides, and the
    counts of the joined script, the reverse side's operations from its far
    end on, then the forward side's."""
    m, nl = gz.blosum62()
    lead, qlen, hq, hd = (int(x) for x in job)
    s0, a0, b0, rev, _ = oracle_py.gapped_one_side(
        "oracle", q, lead + hq - 1, hq - 1, d, hd - 1, DELIM, True, m, nl, gap_open, gap_ext,
        cutoff, traceback=True)
    s1, a1, b1, fwd, _ = oracle_py.gapped_one_side(
        "oracle", q, lead + hq, qlen - hq, d, hd, DELIM, False, m, nl, gap_open, gap_ext, cutoff,
        traceback=True)
    script = rev[::-1] + fwd
    qp, dp, mismatches, opens, extensions, prev = lead + hq - 1 + a0, hd - 1 + b0, 0, 0, 0, SUB
    for op in script:
        if op == SUB:
            mismatches += q[qp] != d[dp]
        elif op != prev:
            opens += 1
        else:
            extensions += 1
        qp, dp, prev = qp + (op != GAP0), dp + (op != GAP1), op
    return (s0 + s1, hq - 1 + a0, hd - 1 + b0, hq + a1, hd + b1, len(script), int(mismatches),
            opens, extensions)


def off_the_waves(jobs):
    """The same jobs, framed so that they take a lane each."""
    part = jobs.copy()
    part[:, 1] -= 1
    return part


def check_against_oracle(q, d, jobs, most, cutoff, gap_open, gap_ext):
    """Every field against the oracle's script, and the flags against the
    form of a lane per result; the share of results without a flag."""
    out = build(q, d, jobs, most, cutoff, gap_open, gap_ext)
    lanes = build(q, d, off_the_waves(jobs), most, cutoff, gap_open, gap_ext)
    assert np.array_equal(out[:, 9], lanes[:, 9])
    served = 0
    for k, job in enumerate(jobs):
        if out[k, 9]:
            continue
        served += 1
        got = tuple(int(x) for x in out[k, :9].astype(np.int64))
        want = by_oracle(q, d, job, cutoff, gap_open, gap_ext)
        assert got == want, (k, job, got, want)
    return served / len(jobs)


# sides that end inside the 64-column window, at its edge and past it; bands
# that stay in the 128- and 256-column windows and that outgrow them (the last
# go to the lanes)
@pytest.mark.parametrize("cutoff,lengths", [
    (52, (1, 2, 3, 12, 13, 24, 25, 49, 61, 62, 63, 64, 65, 66, 67)),
    (52, (125, 126, 127, 128, 129, 130, 400)), (26, (30, 64, 300)), (8, (30, 90)), (0, (20,)),
    (75, (64, 128, 300)), (120, (62, 64, 126, 128, 254, 256, 500, 900))])
@pytest.mark.parametrize("at", [None, 0.0, 1.0])
def test_waves_vs_host(cutoff, lengths, at):
    rng = np.random.default_rng(cutoff + len(lengths))
    print("traceback waves: cutoff", cutoff, "lengths", lengths, "seed", at, flush=True)
    q, d, jobs, most = jobs_of(rng, np.repeat(lengths, 16), (0.3, 1.0), 0.05, at)
    out = build(q, d, jobs, most, cutoff)
    for k, job in enumerate(jobs):
        if out[k, 9] & OVERFLOW:  # 500 rows of bands past 130 columns fill the arena
            assert cutoff == 120 and job[1] * 230 > 1 << 16
            continue
        host = on_host(q, d, job, cutoff)
        assert out[k, 9] == host[9], (k, job, out[k], host)
        if not host[9]:
            assert np.array_equal(out[k], host), (k, job, out[k], host)


@pytest.mark.parametrize("cutoff", [12, 20, 26])
def test_stale_results_are_flagged(cutoff):
    """Inputs on which a few paths read bytes that the extension did not
    write: flagged where the host flags them, and where the form of a lane per
    result does."""
    rng = np.random.default_rng(cutoff)
    print("traceback stale: cutoff", cutoff, flush=True)
    q, d, jobs, most = jobs_of(rng, np.repeat((60, 150, 400), 130), (0.2, 1.0), 0.12)
    out = build(q, d, jobs, most, cutoff)
    host = np.array([on_host(q, d, job, cutoff) for job in jobs])
    assert np.array_equal(out[:, 9], host[:, 9])
    assert (host[:, 9] == STALE).sum() >= 2 and not (host[:, 9] & OVERFLOW).any()
    fresh = host[:, 9] == 0
    assert np.array_equal(out[fresh], host[fresh])
    lanes = build(q, d, off_the_waves(jobs), most, cutoff)
    assert np.array_equal(out[:, 9], lanes[:, 9]) and np.array_equal(out[fresh], lanes[fresh])


@pytest.mark.parametrize("cutoff,gap_open,gap_ext", [
    (52, 11, 1), (60, 0, 3), (35, 8, 0), (52, 5, 2), (120, 30, 1), (10, 11, 1)])
def test_waves_vs_oracle(cutoff, gap_open, gap_ext):
    """Other gap costs: every field and the flags."""
    rng = np.random.default_rng(cutoff + 3 * gap_open)
    print("traceback waves: cutoff", cutoff, "gaps", gap_open, gap_ext, flush=True)
    q, d, jobs, most = jobs_of(rng, np.repeat((40, 63, 64, 130, 260), 20), (0.4, 1.0), 0.04)
    assert check_against_oracle(q, d, jobs, most, cutoff, gap_open, gap_ext) > 0.5


@pytest.mark.parametrize("cutoff,gap_open,gap_ext", [
    (70, 11, 1), (90, 11, 1), (99, 11, 1), (60, 6, 1), (52, 11, 0), (120, 2, 3)])
def test_wide_bands_vs_oracle(cutoff, gap_open, gap_ext):
    """Rows that a gap fills past the window: the side starts again in the
    wider one, sides that the widest one ends and sides that it does not."""
    rng = np.random.default_rng(cutoff + gap_open)
    print("traceback wide bands: cutoff", cutoff, "gaps", gap_open, gap_ext, flush=True)
    q, d, jobs, most = jobs_of(rng, np.repeat((120, 200, 252, 255, 256, 260, 300), 12), (0.3, 1.0),
                               0.04, 0.0)
    assert check_against_oracle(q, d, jobs, most, cutoff, gap_open, gap_ext) > 0.5


def test_more_jobs_than_waves():
    """Jobs past the resident waves' first ones, and their order in the call."""
    rng = np.random.default_rng(5)
    q, d, jobs, most = jobs_of(rng, rng.integers(2, 150, 700), (0.3, 1.0), 0.05)
    pick = rng.integers(0, len(jobs), 30011)
    print("traceback waves:", len(pick), "jobs", flush=True)
    one, many = build(q, d, jobs, most, 52), build(q, d, jobs[pick], most, 52)
    assert np.array_equal(one[pick], many)
    assert np.array_equal(one[:1], build(q, d, jobs[:1], most, 52))


def test_bounds_of_the_call():
    """Subjects longer than described: flagged once a side has more rows than
    described; a longest query that is too small: sides of up to 62 residues
    are built, longer ones flagged; a window of a query (no delimiter where
    its frame ends) is built as before."""
    rng = np.random.default_rng(6)
    q, d, jobs, most = jobs_of(rng, np.repeat((30, 61, 200), 40), (0.9, 1.0), 0.0, 0.0)
    full = build(q, d, jobs, most, 52)
    print("traceback bounds", flush=True)
    few = build(q, d, jobs, 40, 52)
    long = jobs[:, 1] > 100
    assert np.array_equal(few[:40], full[:40])
    assert (few[long, 9] & OVERFLOW).all() and (few[long, :9] == 0).all()
    small = build(q, d, jobs, most, 52, max_query=20)
    assert np.array_equal(small[~long], full[~long])
    assert (small[long, 9] & OVERFLOW).all()
    part = jobs.copy()
    part[:, 1] -= 3  # the frame ends before the query's delimiter
    assert np.array_equal(build(q, d, part, most, 52), full)


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("lengths,n", [((20, 60), 9001), ((200, 400), 3001), ((200, 400), 33)])
def test_jobs_off_the_waves(lengths, n):
    """Jobs that take a lane each, in the waves' scratch where it has room for
    them (long sides) and in a block of their own where not (short ones): all,
    some and one of a call, and a cutoff that the waves do not serve.  Between
    calls no more is kept than the pool's 512 MB."""
    rng = np.random.default_rng(n)
    q, d, jobs, most = jobs_of(rng, rng.integers(*lengths, 200), (0.4, 1.0), 0.04)
    jobs = jobs[rng.integers(0, len(jobs), n)]
    print("traceback lanes: jobs", n, "lengths", lengths, flush=True)
    before = free_bytes()
    full = build(q, d, jobs, most, 52)
    for every in (1, 40, n):
        part = jobs.copy()
        part[::every] = off_the_waves(jobs[::every])
        assert np.array_equal(build(q, d, part, most, 52), full)
    large = build(q, d, jobs, most, 130)
    assert np.array_equal(large[:20], np.concatenate(
        [build(q, d, jobs[k:k + 1], most, 130, max_query=int(jobs[:, 1].max()))
         for k in range(20)]))
    assert before - free_bytes() <= (512 << 20) + (64 << 20)  # and the runtime's own


def test_kept_workspace_is_released():
    rng = np.random.default_rng(9)
    q, d, jobs, most = jobs_of(rng, rng.integers(200, 400, 3000), (0.4, 1.0), 0.04)
    print("traceback: kept workspace", flush=True)
    gz.check(gz.lib().gz_release_workspaces())
    want = build(q, d, jobs, most, 52)
    kept = free_bytes()
    gz.check(gz.lib().gz_release_workspaces())
    assert free_bytes() - kept > 100 << 20
    gz.check(gz.lib().gz_release_workspaces())  # nothing to free
    assert np.array_equal(build(q, d, jobs, most, 52), want)


def test_concurrent_calls():
    """Calls of several threads at once, of different sizes: each has a
    workspace of its own, the kept one or a new one."""
    rng = np.random.default_rng(7)
    sets = [jobs_of(rng, rng.integers(2, most, n), (0.3, 1.0), 0.05)
            for n, most in ((1500, 60), (40, 400), (600, 200))]
    want = [build(q, d, jobs, most, 52) for q, d, jobs, most in sets]
    print("traceback: three threads", flush=True)
    bad = []

    def work(i):
        q, d, jobs, most = sets[i]
        for _ in range(5):
            if not np.array_equal(build(q, d, jobs, most, 52), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_many_short_results_take_lanes():
    """One call of more than 131,072 read results runs a lane each in an
    aligner; the batched form's blocks of the same search run on waves.  The
    outputs are byte-identical."""
    import synthetic
    q, d = synthetic.translated_workload(8, 20000, 24000)
    queries, database = gz.Queries(*q, translated=True), gz.Database(*d)
    print("traceback: one large call and its blocks", flush=True)
    one, st = gz.Aligner(database).align(queries)
    blocks, _ = gz.Aligner(database, batched=1).align(queries)
    assert st["results"] > 131072
    assert one == blocks
