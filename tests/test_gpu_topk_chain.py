"""The top-k batch's device chains: the short one for few queries (every
survivor takes its own waves, the merge reads the pairs), the one with a job
list and the same merge, and the lists a query with more survivors than that
merge sorts falls back to; queries uploaded in one part and in several; no
survivor at all, more results asked for than trajectories.  Answers of every
route equal the host-built path's, and sampled rows the oracle's."""
import time

import numpy as np
import pytest

import oracle as O
from gat_amd import _native as N, api, workloads as W

from tests.devbuf import DevBuf

pytestmark = pytest.mark.gpu
EPS = 5e-4


def _near(seed, n, lengths, spread):
    """Trajectories around one spot: `spread` decides how many boxes touch."""
    db = api.synth_walks(seed, np.asarray(lengths, np.int32)[np.arange(n) % len(lengths)], step_sigma=2e-5)
    off = db.offsets
    rng = np.random.default_rng(seed)
    at = (0.5 + rng.uniform(-spread, spread, (n, 2))).astype(np.float32)
    for i in range(n):
        s = slice(off[i], off[i + 1])
        db.lon[s] += at[i, 0] - db.lon[off[i]]
        db.lat[s] += at[i, 1] - db.lat[off[i]]
    return db


def _check(g, db, q, k, eps, oracle_rows=()):
    ids, dists, st = g.similarity_batched(q, k, eps)
    assert st["pairs"] + st["pruned"] == q.ntraj * db.ntraj
    g.set_topk_device_chain(False)
    hi, hd, hst = g.similarity_batched(q, k, eps)
    g.set_topk_device_chain(True)
    assert (ids == hi).all() and (dists == hd).all()
    assert st["pairs"] == hst["pairs"] and st["cells"] == hst["cells"]
    tid = np.arange(1, db.ntraj + 1, dtype=np.int32)
    for i in oracle_rows:
        oi, od = O.topk(O.edr_batch(q.xy(i + 1), db, eps, nthreads=4), tid, k)
        n = len(oi)
        assert (ids[i][:n] == oi).all() and (dists[i][:n] == od).all(), i
    return st


@pytest.mark.parametrize("nq", [1, 13, 32, 33, 300])
@pytest.mark.parametrize("waves", [1, 2, 4, 8])
def test_chains(gpu, nq, waves):
    rng = np.random.default_rng(nq)
    db = _near(3, 1500, [1, 20, 64, 65, 130, 300, 900], 0.008)
    g = api.GridIndex(W.UNIT_BOX, 0.01, 256).build(db)
    g.set_edr_waves(waves)
    q = _near(100 + nq, nq, rng.choice([1, 16, 63, 64, 129, 600, 1500], nq), 0.005)
    st = _check(g, db, q, 10, EPS, (0, nq - 1))
    assert st["pairs"] > 0
    far = api.TrajSet(q.offsets, q.lon + np.float32(0.4), q.lat)
    assert _check(g, db, far, 10, EPS, (0,))["pairs"] == 0
    _check(g, db, q, 10, EPS)  # the first batch again, after one without survivors
    g.set_edr_waves(4)


@pytest.mark.parametrize("nq", [3, 40])
def test_many_survivors(gpu, nq):
    """1,024 survivors of a query are the most the merge sorts; one more sends
    the batch to the lists, and a small batch over its pairs to the job list."""
    for n in (1023, 1024, 1025):
        db = _near(5, n, [12, 20], 1e-4)
        g = api.GridIndex(W.UNIT_BOX, 0.01, 256).build(db)
        q = _near(6, nq, [14], 1e-4)
        for _ in range(2):  # the second with the survivors of the first known
            assert _check(g, db, q, 5, 0.01, (0,))["pairs"] == nq * n


def test_more_results_than_trajectories_and_upload_parts(gpu):
    db = _near(7, 9, [40, 3], 1e-3)
    g = api.GridIndex(W.UNIT_BOX, 0.01, 256).build(db)
    q = _near(8, 2, [30], 1e-3)
    for k in (1, 9, 30):
        ids, dists, _ = g.similarity_batched(q, k, EPS)
        full = O.edr_batch(q.xy(1), db, EPS, nthreads=4)
        oi, od = O.topk(full, np.arange(1, 10, dtype=np.int32), k)
        assert (ids[0][:len(oi)] == oi).all() and (dists[0][:len(od)] == od).all()
    # 600,000 points go up in several parts, whose borders fall on trajectories.
    many = _near(9, 400, [1500], 1e-3)
    _check(g, db, many, 4, EPS, (0, 399))


# (candidates' lengths, query length, k): the cut's ties found by reading ids in
# order (common ties, and ones hidden behind ids in length order), by gathering
# their lists' entries (a rare tie), and by searching over lists too many or too
# long to gather; fewer candidates than a round reads; k of one and of the most.
def _sizes(case):
    rng = np.random.default_rng(11)
    if case == "common":
        return rng.integers(1, 700, 30000), 511, 50
    if case == "few":
        return rng.integers(1, 30, 100), 16, 100
    if case == "one":
        return rng.integers(1, 300, 5000), 64, 1
    if case == "hidden":  # 45,000 of 120,000 at the cut, all behind the first 65,536 ids
        return np.sort(np.concatenate([np.full(75000, 2000), rng.integers(480, 512, 45000)]))[::-1], 511, 1024
    if case == "rare":
        n = np.full(60000, 1900)
        n[rng.choice(60000, 80, False)] = 100
        return n, 100, 50
    if case == "lists":  # 17,000 entries, more than are gathered
        n = np.full(600000, 2000)
        n[rng.choice(600000, 17000, False)] = rng.integers(260, 512, 17000)
        return n, 511, 1024
    raise KeyError(case)


@pytest.mark.parametrize("case", ["common", "few", "one", "hidden", "rare", "lists"])
@pytest.mark.parametrize("nsurv", [0, 1, 300])
def test_merge_routes(gpu, case, nsurv):
    h = N.hip()
    clen, a, k = _sizes(case)
    clen = np.ascontiguousarray(clen, np.int32)
    nc, w = len(clen), api.MAX_TRAJ_LEN + 1
    rng = np.random.default_rng(nsurv)
    table, by_len = DevBuf(w * w * 4), DevBuf(w * w * 4)
    N.check_hip(h.gat_edr_mismatch_table(w - 1, table.ptr, None))
    N.check_hip(h.gat_edr_length_table(table.ptr, w, by_len.ptr, None))
    F = table.get(np.int32, w * w).reshape(w, w)
    assert (by_len.get(np.int32, w * w).reshape(w, w) == np.triu(F) + np.triu(F, 1).T).all()
    d = F[np.minimum(a, clen), np.maximum(a, clen)].astype(np.int64)
    kk = min(k, nc)
    # Survivors below, at and above the cut, some among the ties' first ids.
    nsurv = min(nsurv, nc // 4)
    sid = np.sort(rng.choice(min(nc, 4000), nsurv, False)).astype(np.int32)
    cut = np.sort(d)[kk - 1]
    d[sid] = np.clip(cut + rng.integers(-2, 3, nsurv), 0, 2 * (w - 1))
    order = np.lexsort((np.arange(nc), d))[:kk]
    len_ids = np.argsort(clen, kind="stable").astype(np.int32)
    len_off = np.concatenate([[0], np.cumsum(np.bincount(clen, minlength=w))]).astype(np.int32)
    qlen, dclen = DevBuf.of(np.array([a], np.int32)), DevBuf.of(clen)
    ids, offs = DevBuf.of(len_ids), DevBuf.of(len_off)
    mix = rng.permutation(nsurv)
    pairs = np.zeros((max(nsurv, 1), 2), np.int32)
    pairs[:nsurv, 1] = sid[mix]
    dist = np.zeros(max(nsurv, 1), np.int32)
    dist[:nsurv] = d[sid[mix]]
    dpairs, ddist = DevBuf.of(pairs), DevBuf.of(dist)
    out_i, out_d = DevBuf(4 * k), DevBuf(4 * k)
    ctl0 = np.zeros(32, np.uint32)
    ctl0[0] = nsurv
    ctl, back = DevBuf.of(ctl0), DevBuf(34 * 4)
    N.check_hip(h.gat_edr_merge(by_len.ptr, w, qlen.ptr, 1, dclen.ptr, nc, ids.ptr, offs.ptr, dpairs.ptr, ddist.ptr,
                                max(nsurv, 1), k, kk, out_i.ptr, out_d.ptr, ctl.ptr, back.ptr, None, None))
    words = back.get(np.uint32, 34)
    assert words[0] == nsurv and words[2] == 0 and words[3] == 0
    assert (out_i.get(np.int32, kk) == order + 1).all() and (out_d.get(np.int32, kk) == d[order]).all()
    # The lists' form of the same merge.
    start = DevBuf.of(np.array([0, nsurv], np.int32))
    lid = DevBuf.of(np.concatenate([sid, [0]]).astype(np.int32))
    ldist = DevBuf.of(np.concatenate([d[sid], [0]]).astype(np.int32))
    status = DevBuf.of(np.array([7], np.int32))
    N.check_hip(h.gat_edr_topk(table.ptr, w, qlen.ptr, 1, dclen.ptr, nc, ids.ptr, offs.ptr, start.ptr, lid.ptr,
                               ldist.ptr, k, kk, out_i.ptr, out_d.ptr, status.ptr, None))
    assert status.get(np.int32, 1)[0] == 0
    assert (out_i.get(np.int32, kk) == order + 1).all() and (out_d.get(np.int32, kk) == d[order]).all()


@pytest.mark.parametrize("nq", [13, 200])  # the short chain and the job-list chain
def test_stage_times_add_up(gpu, nq):
    """Each stage's device time is what it can be, batch after batch: the merge's
    start is written by another workgroup than the one that brings the rest of
    the clock readings back, and a stale reading would wrap around."""
    db = api.synth_walks(3, api.synth_lengths(3, 4000, "lognormal", 64, 0.8, 8, 512))
    g = api.GridIndex(W.UNIT_BOX, 0.01, 64).build(db)
    q = api.synth_queries(5, api.synth_lengths(4, nq, "uniform", 16, 256, 16, 256), db, copy_mode=2)
    g.similarity_batched(q, 20, EPS)
    for _ in range(100):
        t0 = time.perf_counter()
        st = g.similarity_batched(q, 20, EPS)[2]
        wall = (time.perf_counter() - t0) * 1e3
        stages = [st["filter_ms"], st["kernel_ms"], st["merge_ms"]]
        assert min(stages) > 0 and sum(stages) <= wall, (stages, wall)


def test_filter_time_leaves_out_the_job_list(gpu):
    """filter_ms is the filter's on the device chain as on the host-built path,
    where events bracket it: in a batch whose 90,000 survivors keep the one
    workgroup of the job list busy several times as long."""
    db = _near(21, 300, [40, 60], 1e-4)
    g = api.GridIndex(W.UNIT_BOX, 0.01, 64).build(db)
    q = _near(22, 300, [40, 60], 1e-4)
    ms = {}
    for chain in (True, False):
        g.set_topk_device_chain(chain)
        runs = [g.similarity_batched(q, 20, EPS)[2] for _ in range(6)]
        assert runs[0]["pairs"] > 80_000
        ms[chain] = min(r["filter_ms"] for r in runs[2:])
    assert ms[True] <= 1.25 * ms[False] + 0.01, ms
