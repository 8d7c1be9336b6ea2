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


@pytest.mark.parametrize("kind", [0, 1, 2])  # FSG, the GT-quadtree, STIG
def test_a_small_workspace_discards_no_other(gpu, layout, kind):
    """One index's part of a group has one rectangle more than its workspace was
    sized for: that index runs step by step and the others' queued pipelines
    are used.  A part that outgrows a capacity is the only one run again."""
    db = api.synth_walks(9, api.synth_lengths(9, 2500, "uniform", 1, 90, 1, 90), step_sigma=4e-3)
    ix = (api.GridIndex(W.UNIT_BOX, 0.01, 64).build(db), api.StigIndex(64).build(db),
          api.FsgIndex(W.UNIT_BOX, 0.01).build(db))
    for i in ix:
        i.set_result_layout(layout)
    m = api.MixedRange(*ix)
    rng = np.random.default_rng(kind)
    sides = [(1e-4, 9e-4), (2e-3, 2e-2), (4e-2, 6e-2)]  # an index each

    def run(counts, lo_hi):
        rects = np.concatenate([_rects(rng, n, *s) for n, s in zip(counts, lo_hi)])
        c, d, route, _ = m.run(rects, 1e-6, 1e-3)
        assert (np.bincount(route, minlength=3) == counts).all()
        want_c, want_d = _expected(ix, rects, route)
        assert (c == want_c).all() and (d == want_d).all()
        return np.array(list(m.pipelines().values()))

    counts = np.array([300, 300, 300])
    assert run(counts, sides).tolist() == [0, 3, 0]
    counts[kind] += 1
    assert run(counts, sides).tolist() == [2, 4, 0]
    sides[2] = (0.4, 0.6)  # STIG's rectangles outgrow its lists
    assert run(counts, sides).tolist() == [5, 5, 1]


@pytest.mark.parametrize("run_indexed", [True, False])
def test_digest_time_is_the_digests(gpu, run_indexed):
    """digest_ms of a queued group covers the digest kernels, which cannot read
    the pairs faster than the memory's 8 TB/s."""
    db = api.synth_walks(9, api.synth_lengths(9, 40_000, "uniform", 16, 256, 16, 256), step_sigma=4e-3)
    ix = (api.GridIndex(W.UNIT_BOX, 0.01, 256).build(db, device=True), api.StigIndex(256).build(db, device=True),
          api.FsgIndex(W.UNIT_BOX, 0.01).build(db, device=True))
    for i in ix:
        i.set_result_layout(run_indexed)
    m = api.MixedRange(*ix)
    rects = _rects(np.random.default_rng(1), 600, 0.24, 0.26)
    for _ in range(2):
        st = m.run(rects)[3]
    assert m.pipelines() == {"queued": 1, "stepped": 1, "discarded": 0}
    assert st["pairs"] > 1e8 and st["digest_ms"] * 1e-3 >= 8 * st["pairs"] / 8e12, st


def test_batched_form_over_growing_batches(indexes):
    rng = np.random.default_rng(5)
    for ix in indexes:
        for lo, hi, n in ((1e-3, 2e-2, 400), (1e-3, 2e-2, 300), (1e-2, 5e-1, 700), (1e-3, 2e-2, 257)):
            rects = _rects(rng, n, lo, hi)
            b, p = ix.range_batched(rects), ix.range_pairs(rects)
            assert (np.asarray(b.counts()) == np.asarray(p.counts())).all()
            assert (np.asarray(b.digests()) == np.asarray(p.digests())).all()
