"""Groups of a mixed run that are queued on the three indexes' streams with one
wait (another shape than the captured one, or too few groups to capture):
answers against each index's own plain form, on a first run, on one whose
workspaces earlier runs have sized, after small batches sized them for less, and
with one index left out of a group, in both result layouts (a queued or replayed
group that outgrows its pair buffer has its digests queued behind it); and the
single index's batched form without a graph over batches that grow and shrink."""
import numpy as np
import pytest

from gat_amd import api, workloads as W

pytestmark = pytest.mark.gpu


def _rects(rng, n, lo, hi):
    c = rng.random((n, 2)).astype(np.float32)
    s = np.exp(rng.uniform(np.log(lo), np.log(hi), n)).astype(np.float32)
    return np.concatenate([c - s[:, None] / 2, c + s[:, None] / 2], 1).astype(np.float32)


@pytest.fixture(scope="module")
def indexes(gpu):
    db = api.synth_walks(9, api.synth_lengths(9, 2500, "uniform", 1, 90, 1, 90), step_sigma=4e-3)
    return (api.GridIndex(W.UNIT_BOX, 0.01, 64).build(db), api.StigIndex(64).build(db),
            api.FsgIndex(W.UNIT_BOX, 0.01).build(db))


def _expected(indexes, rects, route):
    g, s, f = indexes
    per = []
    for ix in (f, g, s):
        b = ix.range_pairs(rects)
        per.append((np.asarray(b.counts()), np.asarray(b.digests())))
    pick = lambda k: np.choose(route, [p[k] for p in per])
    return pick(0), pick(1)


@pytest.fixture(params=[True, False], ids=["runs", "regions"])
def layout(indexes, request):
    for ix in indexes:
        ix.set_result_layout(request.param)
    yield request.param
    for ix in indexes:
        ix.set_result_layout(True)


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("group", [300, 2000])  # several groups of two shapes, and one group
def test_queued_groups(indexes, layout, graph, group):
    g, s, f = indexes
    rng = np.random.default_rng(group)
    m = api.MixedRange(g, s, f)
    for lo, hi, n in ((1e-3, 5e-2, 1000), (1e-3, 5e-2, 1000), (1e-2, 4e-1, 1000), (1e-3, 5e-2, 999), (1e-3, 2e-3, 700)):
        rects = _rects(rng, n, lo, hi)
        counts, digests, route, st = m.run(rects, 1e-5, 1e-3, group_size=group, graph=graph)
        c, d = _expected(indexes, rects, route)
        assert (counts == c).all() and (digests == d).all(), (lo, hi, n)
        assert st["pairs"] == int(c.astype(np.int64).sum())


def test_batched_form_over_growing_batches(indexes):
    rng = np.random.default_rng(5)
    for ix in indexes:
        for lo, hi, n in ((1e-3, 2e-2, 400), (1e-3, 2e-2, 300), (1e-2, 5e-1, 700), (1e-3, 2e-2, 257)):
            rects = _rects(rng, n, lo, hi)
            b, p = ix.range_batched(rects), ix.range_pairs(rects)
            assert (np.asarray(b.counts()) == np.asarray(p.counts())).all()
            assert (np.asarray(b.digests()) == np.asarray(p.digests())).all()
