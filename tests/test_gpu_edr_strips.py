"""The EDR sweep's strips (one, two or four rows per lane, the remainder rule
between them), its blocks that test no match because the strip's box and the
block's columns lie apart, and the capture of D[n][m] in both kinds of block:
every kernel form (plain handler, 16- and 64-lane segments, several waves per
pair) against the oracle's row-major restatement of Grid.cpp:1222-1318."""
import numpy as np
import pytest

import oracle as O
from gat_amd import api, workloads as W

pytestmark = pytest.mark.gpu
EPS = 5e-4


def _commuter(rng, n, homes):
    """A trajectory that stays at one of a few places for a stretch and jumps
    to another, so blocks of both kinds alternate; a few NaN and infinite
    points, which match nothing."""
    xy = np.empty((n, 2), np.float32)
    at = 0
    while at < n:
        k = int(rng.integers(3, 70))
        xy[at:at + k] = homes[rng.integers(len(homes))] + rng.normal(0, 3e-4, (min(k, n - at), 2))
        at += k
    if n > 40:
        bad = rng.integers(0, n, 3)
        xy[bad[0], 0] = np.nan
        xy[bad[1]] = np.nan
        xy[bad[2], 1] = np.inf
    return xy.astype(np.float32)


def _set(xys):
    lens = [len(x) for x in xys]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    xy = np.concatenate(xys)
    return api.TrajSet(off, np.ascontiguousarray(xy[:, 0]), np.ascontiguousarray(xy[:, 1]))


def _want(q, db, pairs):
    return np.array([O.edr(q.xy(a + 1), db.xy(b + 1), EPS) for a, b in pairs], np.int32)


# Rows per strip: 16 or 64 lanes of 4, 2 and 1 rows, and what the remainder rule makes of three.
ROWS16 = [1, 15, 16, 17, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 96, 112, 113, 128]
ROWS64 = [192, 193, 255, 256, 257, 320, 384, 448, 449, 512, 513, 1024, 1025, 2047, 2048]


@pytest.mark.parametrize("lengths,others", [(ROWS16, [16, 31, 64, 130, 256]), (ROWS64, [192, 257, 700, 2048])])
def test_strips_against_the_oracle(gpu, lengths, others):
    rng = np.random.default_rng(len(lengths))
    homes = np.array([[0.2, 0.2], [0.2005, 0.2], [0.7, 0.3], [0.71, 0.31]])
    store = [_commuter(rng, n, homes) for n in lengths]
    # One trajectory with no point near any other: every block of its pairs is far.
    store.append(np.full((lengths[-1] // 2 + 1, 2), 0.95, np.float32))
    queries = [_commuter(rng, n, homes) for n in others]
    # The index needs points inside its box; the distances read the queries as they are.
    clean = [np.where(np.isfinite(x), x, np.float32(0.5)) for x in store]
    db, q = _set(clean), _set(queries)
    g = api.GridIndex(W.UNIT_BOX, 0.01, 256).build(db)
    pairs = np.array([(a, b) for a in range(q.ntraj) for b in range(db.ntraj)], np.int32)
    want = _want(q, db, pairs)
    plain = np.concatenate([g.edr_all(q.xy(a + 1), EPS) for a in range(q.ntraj)])
    assert (plain == want).all(), "plain handler"
    for split in (2048, 1):  # 16-lane segments for every pair; one wave (or several) per pair
        g.set_edr_params(split)
        for waves in (1, 2, 4, 8) if split == 1 else (1,):
            g.set_edr_waves(waves, every_long_pair=True)
            got, _ = g.edr_batched_pairs(q, pairs, EPS)
            bad = np.nonzero(got != want)[0]
            assert len(bad) == 0, (split, waves, [(pairs[i].tolist(), int(got[i]), int(want[i])) for i in bad[:8]])
