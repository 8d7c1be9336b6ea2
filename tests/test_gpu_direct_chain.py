"""The direct form's device chain and the gathered readback: batches of every
size around a wave's four entries and the regions kernel's 256 threads, batches
that outgrow the pairs and the selection's list, leaves of more points than one
round takes, rectangles that select nothing; counts, digests and pair sets
against the plain path and inclusive brute force.  (Stores of unpacked ids:
test_unpacked_ids of test_gpu_build.py.)"""
import threading

import numpy as np
import pytest

import oracle as O
from gat_amd import api, workloads as W

pytestmark = pytest.mark.gpu


def _rects(rng, n):
    c = rng.random((n, 2)).astype(np.float32)
    s = np.exp(rng.uniform(np.log(1e-4), np.log(0.3), n)).astype(np.float32)
    r = np.concatenate([c - s[:, None] / 2, c + s[:, None] / 2], 1).astype(np.float32)
    if n > 2:
        r[0] = [2, 2, 3, 3]  # outside the domain
        r[1] = [0.5, 0.5, 0.4, 0.4]  # inverted
    return r


@pytest.mark.parametrize("nq", [1, 3, 4, 5, 255, 256, 257, 700])
@pytest.mark.parametrize("leaf", [64, 700])  # one round of 256 points per entry, and three
def test_direct_chain(gpu, nq, leaf):
    rng = np.random.default_rng(nq)
    db = api.synth_walks(5, api.synth_lengths(5, 1500, "uniform", 1, 90, 1, 90), step_sigma=4e-3)
    rects = _rects(rng, nq)
    want_c, want_d = O.brute_range(db, rects, "digest", nthreads=8)
    for ix in (api.GridIndex(W.UNIT_BOX, 0.02, leaf), api.StigIndex(leaf), api.FsgIndex(W.UNIT_BOX, 0.05)):
        ix.build(db).set_batch_params(32, 1 << 20)
        plain = ix.range_pairs(rects)
        pc, pd, pp = plain.counts(), plain.digests(), plain.per_query()
        if not isinstance(ix, api.GridIndex):  # the GT-quadtree's touching test is strict
            assert (pc == want_c).all() and (pd == want_d).all()
        for _ in range(2):  # the first call grows the buffers, the second finds them
            res = ix.range_batched(rects)
            assert res.pairs_total == plain.pairs_total and res.candidates == plain.candidates
            assert (res.counts() == pc).all() and (res.digests() == pd).all()
            for a, b in zip(res.per_query(), pp):
                assert sorted(map(tuple, a.tolist())) == sorted(map(tuple, b.tolist()))
        # Leaf-major batches read back through their runs.
        res = ix.set_batch_params(8, 0).range_batched(rects)
        assert (res.counts() == pc).all()
        for a, b in zip(res.per_query(), pp):
            assert sorted(map(tuple, a.tolist())) == sorted(map(tuple, b.tolist()))


def test_direct_outgrows_the_list(gpu):
    """More (leaf, rectangle) entries than the list's first 65,536: it grows and
    the batch runs again, and the next one of its size fits."""
    db = api.synth_walks(6, np.full(3000, 60, np.int32), step_sigma=4e-3)
    ix = api.GridIndex(W.UNIT_BOX, 0.005, 16).build(db)
    rects = np.tile(np.array([[0.0, 0.0, 1.0, 1.0]], np.float32), (40, 1))
    rects[1::2] = [0.25, 0.25, 0.75, 0.75]
    plain = ix.range_pairs(rects)
    pc, pd = plain.counts(), plain.digests()
    # The leaf-major form counts the entries.
    assert ix.set_batch_params(32, 0).range_batched(rects).leaf_queries > 1 << 16
    fresh = api.GridIndex(W.UNIT_BOX, 0.005, 16).build(db)
    for _ in range(2):
        res = fresh.range_batched(rects)
        assert res.leaf_queries > 1 << 16
        assert (res.counts() == pc).all() and (res.digests() == pd).all()


@pytest.mark.parametrize("direct", [256, 0])  # regions of the direct form, runs of the leaf-major one
def test_a_batch_read_by_several_threads(gpu, direct):
    """Digests and pairs of one batch asked for by several threads at once (a
    reader's call leaves the interpreter while it waits for the device)."""
    db = api.synth_walks(5, api.synth_lengths(5, 3000, "uniform", 1, 90, 1, 90), step_sigma=4e-3)
    ix = api.GridIndex(W.UNIT_BOX, 0.02, 64).build(db).set_batch_params(32, direct)
    res = ix.range_batched(_rects(np.random.default_rng(8), 200))
    counts = np.concatenate([[0], np.cumsum(res.counts(), dtype=np.int64)])

    def keys():
        p = res.pairs().astype(np.int64)
        key = np.repeat(np.arange(len(counts) - 1), np.diff(counts)) << 40 | p[:, 0] << 16 | p[:, 1]
        return np.sort(key)

    want_d, want_k = res.digests(), keys()
    bad = []

    def read(n):
        for _ in range(n):
            if not (res.digests() == want_d).all() or not (keys() == want_k).all():
                bad.append(threading.get_ident())

    threads = [threading.Thread(target=read, args=(40,)) for _ in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
