"""Digest kernels over per-query regions and over runs: odd starts and lengths
around the 16-byte loads and a row's 128 pairs in flight, buffers that are only
8-byte aligned, a region split over several workgroups, more queries than the
LDS sums hold, regions at, across and past the end of the pairs; against the
same mix in numpy."""
import ctypes as C

import numpy as np
import pytest

from gat_amd import _native as N, api

from tests.devbuf import DevBuf

pytestmark = pytest.mark.gpu


def _mix(pairs):
    z = (pairs[:, 0].astype(np.uint32).astype(np.uint64) << np.uint64(32)) | pairs[:, 1].astype(np.uint32)
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


@pytest.mark.parametrize("offset", [0, 1])  # pairs the buffer starts past a 16-byte boundary
@pytest.mark.parametrize("nq", [1, 3, 5000])
def test_digests(gpu, offset, nq):
    rng = np.random.default_rng(nq + offset)
    lens = np.array([0, 1, 2, 3, 31, 32, 33, 127, 128, 129, 255, 500, 4097, 40_000 if nq < 10 else 7])
    count = np.concatenate([lens, rng.integers(0, 40, max(nq, 14))])
    count = count[:nq] if nq >= 14 else np.array([40_001, 1, 129][:nq])
    base = np.cumsum(count + rng.integers(0, 3, nq)) - count  # gaps of 0 to 2 pairs
    total = int(base[-1] + count[-1])
    pairs = rng.integers(0, 2**31, (total, 2)).astype(np.int32)
    dev = DevBuf.of(np.concatenate([np.zeros((offset, 2), np.int32), pairs]))
    ptr = C.c_void_p(dev.ptr.value + 8 * offset)
    out = DevBuf.of(np.full(nq, 7, np.uint64))
    qbase, qcount = DevBuf.of(base.astype(np.uint64)), DevBuf.of(count.astype(np.uint32))
    m = _mix(pairs)
    with np.errstate(over="ignore"):
        want = np.array([m[b:b + c].sum(dtype=np.uint64) for b, c in zip(base, count)], np.uint64)
    N.check_hip(N.hip().gat_pairs_digest(ptr, qbase.ptr, qcount.ptr, nq, total, out.ptr, None))
    N.check_hip(N.hip().gat_device_sync())
    assert (out.get(np.uint64, nq) == want).all()
    # The same regions as runs, each cut in up to three, in shuffled order.
    runs = []
    for q, (b, c) in enumerate(zip(base, count)):
        cut = np.unique(np.concatenate([[0, c], rng.integers(0, c + 1, 2)]))
        runs += [(q, cut[i + 1] - cut[i], b + cut[i]) for i in range(len(cut) - 1)] or [(q, 0, b)]
    runs.append((nq, 1, 0))          # a query outside the batch
    runs.append((0, 2, total - 1))   # pairs past the buffer
    runs = np.array(runs, api.RUN)[rng.permutation(len(runs))]
    drun = DevBuf.of(runs)
    N.check_hip(N.hip().gat_runs_digest(ptr, total, drun.ptr, len(runs), nq, out.ptr, None))
    N.check_hip(N.hip().gat_device_sync())
    assert (out.get(np.uint64, nq) == want).all()


@pytest.mark.parametrize("capacity", [0, 1, 2, 999, 1000])
@pytest.mark.parametrize("offset", [0, 1])
def test_regions_past_the_pairs(gpu, capacity, offset):
    """Regions as a batch leaves them that outgrew its pair buffer: every start
    around the capacity, and far past it, inside a larger allocation."""
    rng = np.random.default_rng(capacity)
    room = 1 << 16
    pairs = rng.integers(0, 2**31, (room, 2)).astype(np.int32)
    dev = DevBuf.of(np.concatenate([np.zeros((offset, 2), np.int32), pairs]))
    base = np.concatenate([np.arange(max(capacity - 40, 0), capacity + 41), np.arange(5000, 5003), [room - 1]])
    base = np.repeat(base, 4).astype(np.uint64)
    count = np.tile([0, 1, 33, 4096], len(base) // 4).astype(np.uint32)
    m = _mix(pairs)
    with np.errstate(over="ignore"):
        want = np.array([m[b:min(b + c, capacity)].sum(dtype=np.uint64) if b < capacity else 0
                         for b, c in zip(base.astype(int), count.astype(int))], np.uint64)
    out = DevBuf.of(np.full(len(base), 7, np.uint64))
    qbase, qcount = DevBuf.of(base), DevBuf.of(count)
    N.check_hip(N.hip().gat_pairs_digest(C.c_void_p(dev.ptr.value + 8 * offset), qbase.ptr, qcount.ptr, len(base),
                                         capacity, out.ptr, None))
    N.check_hip(N.hip().gat_device_sync())
    assert (out.get(np.uint64, len(base)) == want).all()
