"""The bitmap form's device chain (gat_direct_bitmap, gat_bitmap_finish): rows
that end off byte, word and 32-byte borders, batches around one launch's
rectangles, leaves of one round of points and of several, rectangles that
select nothing and everything, a batch that outgrows the selection's list;
against the bitmap of the pair form's results."""
import numpy as np
import pytest

from gat_amd import api, workloads as W

pytestmark = pytest.mark.gpu


def _want(ix, rects, ntraj):
    res = ix.range_pairs(rects)
    want = np.zeros((len(rects), ntraj + 1), np.uint8)
    for i, p in enumerate(res.per_query()):
        want[i, np.asarray(p)[:, 0]] = 1
    return want


@pytest.mark.parametrize("ntraj", [1, 6, 7, 31, 255, 2000])
@pytest.mark.parametrize("nq", [1, 3, 100, 1024, 1025])
def test_bitmap_chain(gpu, ntraj, nq):
    rng = np.random.default_rng(ntraj + nq)
    db = api.synth_walks(5, api.synth_lengths(5, ntraj, "uniform", 1, 90, 1, 90), step_sigma=4e-3)
    c = rng.random((nq, 2)).astype(np.float32)
    s = np.exp(rng.uniform(np.log(1e-4), np.log(0.3), nq)).astype(np.float32)
    rects = np.concatenate([c - s[:, None] / 2, c + s[:, None] / 2], 1).astype(np.float32)
    rects[0] = [0, 0, 1, 1]
    if nq > 2:
        rects[1] = [2, 2, 3, 3]  # outside the domain
        rects[2] = [0.5, 0.5, 0.4, 0.4]  # inverted
    for ix in (api.GridIndex(W.UNIT_BOX, 0.01, 64).build(db), api.GridIndex(W.UNIT_BOX, 0.25, 1024).build(db),
               api.FsgIndex(W.UNIT_BOX, 0.01).build(db), api.StigIndex(700).build(db)):
        want = _want(ix, rects, ntraj)
        for _ in range(2):  # the second over the first's bitmap
            assert (ix.range_bitmap(rects) == want).all()


def test_bitmap_outgrows_the_list(gpu):
    db = api.synth_walks(6, np.full(3000, 60, np.int32), step_sigma=4e-3)
    ix = api.GridIndex(W.UNIT_BOX, 0.005, 16).build(db)
    rects = np.tile(np.array([[0.0, 0.0, 1.0, 1.0]], np.float32), (40, 1))
    want = _want(ix, rects, 3000)
    assert want.sum() > 40 * 2900
    assert (ix.range_bitmap(rects) == want).all()
