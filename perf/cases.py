"""The workloads this framework's speed is measured on.

Every case is one call (or one call and the readback of its answer) that a
program makes over an index it keeps resident: range batches on the GT-quadtree,
MortonGrid, STIG and FSG, the reference's bitmap handler, the batch routed over
three indexes, exact top-k similarity, all-pairs EDR distances, the plain
similarity query, and the construction of an index on the device.  The data are
the seeded random walks of gat_amd.workloads (unit box, step 1e-4): lengths
U{16..256} ("uniform") or lognormal with sigma 0.8 clipped to [8, 2048]
("lognormal", by its median), queries every other one a noisy copy of an indexed
trajectory, eps 5e-4.

Every output is whole numbers (ids, counts, distances) or copied coordinates, so
two correct implementations agree bit for bit.  The pairs of a range batch come
in no order: where a program reads them back, they are returned sorted; where
they stay in HBM for a consumer on the device, the consumer is the index's own
digest pass, which reads every pair, and the per-query counts and digests are
what the serving loop and the routed batch return too.
"""
from __future__ import annotations

import math
import random

import numpy as np

import gat_amd as G

UNIT_BOX = (0.0, 0.0, 1.0, 1.0)
EPS = 5e-4
SIGMA = 0.8

# Largest costs a drawn case may have: the largest listed ones.
MAX_PAIRS = 6.4e8   # result pairs of a range batch
MAX_CELLS = 1.6e10  # cells of the all-pairs EDR case


def listed() -> list[dict]:
    return [
        # The smallest call: one window over a small index, its hits read back.
        {"name": "range_one", "op": "range", "index": "grid", "ntraj": 20_000, "lengths": "uniform", "median": 0,
         "cell": 0.01, "leaf": 256, "nq": 1, "side_lo": 0.01, "side_hi": 0.01, "want": "pairs"},
        # A screenful of windows over STIG, every hit read back.
        {"name": "range_windows", "op": "range", "index": "stig", "ntraj": 20_000, "lengths": "uniform", "median": 0,
         "cell": 0.01, "leaf": 256, "nq": 97, "side_lo": 0.01, "side_hi": 0.01, "want": "pairs"},
        # The reference's own range call: a trajectory bitmap per rectangle on the host.
        {"name": "range_bitmap", "op": "bitmap", "index": "grid", "ntraj": 20_000, "lengths": "uniform", "median": 0,
         "cell": 0.01, "leaf": 256, "nq": 100, "side_lo": 0.01, "side_hi": 0.01},
        # What the serving loop forms out of arriving rectangles: a batch under the direct form's limit.
        {"name": "range_serving", "op": "range", "index": "grid", "ntraj": 1_000_000, "lengths": "lognormal",
         "median": 64, "cell": 0.001, "leaf": 256, "nq": 100, "side_lo": 1e-4, "side_hi": 5e-2, "want": "digests"},
        # The large offline batch: 10k squares over 1M trajectories, the captured pipeline.
        {"name": "range_batch", "op": "range", "index": "grid", "ntraj": 1_000_000, "lengths": "lognormal",
         "median": 64, "cell": 0.001, "leaf": 256, "nq": 10_000, "side_lo": 1e-4, "side_hi": 1e-1, "want": "digests"},
        # Rectangles routed by area over FSG, the GT-quadtree and STIG, hot spots included.
        {"name": "range_mixed", "op": "mixed", "ntraj": 300_000, "lengths": "lognormal", "median": 64,
         "cell": 0.001, "leaf": 256, "nq": 9_001, "side_lo": 1e-4, "side_hi": 1e-1, "group": 2048},
        # One similarity query, as an interactive caller sends it.
        {"name": "topk_one", "op": "topk", "ntraj": 20_000, "lengths": "uniform", "median": 0, "cell": 0.01,
         "nq": 1, "qlen_lo": 128, "qlen_hi": 128, "k": 10},
        # The top-k batches of the serving loop.
        {"name": "topk_serving", "op": "topk", "ntraj": 300_000, "lengths": "lognormal", "median": 64, "cell": 0.001,
         "nq": 13, "qlen_lo": 16, "qlen_hi": 512, "k": 20},
        # The offline top-k batch: 1024 queries against 200k candidates.
        {"name": "topk_batch", "op": "topk", "ntraj": 200_000, "lengths": "lognormal", "median": 128, "cell": 0.001,
         "nq": 1024, "qlen_lo": 16, "qlen_hi": 1024, "k": 50},
        # The distance matrix of a few queries against every trajectory.
        {"name": "edr_all", "op": "edr_all", "ntraj": 60_000, "lengths": "lognormal", "median": 128, "cell": 0.001,
         "nq": 3, "qlen_lo": 64, "qlen_hi": 1024},
        # The reference's top-k call: one 128-point query against every trajectory, no pruning.
        {"name": "similarity", "op": "similarity", "ntraj": 20_000, "lengths": "uniform", "median": 0, "cell": 0.01,
         "nq": 1, "qlen_lo": 128, "qlen_hi": 128, "k": 10},
        # Index construction on the device, the store read back.
        {"name": "build", "op": "build", "index": "grid", "ntraj": 50_000, "lengths": "lognormal", "median": 64,
         "cell": 0.002, "leaf": 256},
    ]


def _most_pairs(case: dict) -> int:
    """The hits of a batch whose rectangles all have the largest side, on evenly spread points."""
    return int(case["nq"] * case["ntraj"] * _mean_length(case) * case["side_hi"] ** 2)


def _log(rng: random.Random, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _mean_length(case: dict) -> float:
    return 136.0 if case["lengths"] == "uniform" else case["median"] * math.exp(SIGMA * SIGMA / 2)


def _mean_area(case: dict) -> float:
    lo, hi = case["side_lo"], case["side_hi"]
    return lo * lo if hi <= lo else (hi * hi - lo * lo) / (2 * math.log(hi / lo))


def _database(rng: random.Random, ntraj_lo: int, ntraj_hi: int) -> dict:
    ntraj = int(_log(rng, ntraj_lo, ntraj_hi))
    kind = rng.choice(["uniform", "lognormal"])
    return {"ntraj": ntraj, "lengths": kind, "median": rng.choice([64, 96, 128]) if kind == "lognormal" else 0}


def _cell(rng: random.Random, ntraj: int) -> float:
    # About a leaf's worth of points in a handful of cells, as the configurations have it.
    return rng.choice([0.01, 0.005]) if ntraj < 60_000 else rng.choice([0.002, 0.001])


def draw(rng: random.Random) -> dict:
    op = rng.choice(["range", "range", "range", "bitmap", "mixed", "topk", "topk", "edr_all", "similarity", "build"])
    if op == "range":
        c = {"op": op, "index": rng.choice(["grid", "grid", "mgrid", "stig", "fsg"]), **_database(rng, 20_000, 900_000)}
        c.update(cell=_cell(rng, c["ntraj"]), leaf=rng.choice([128, 256, 500]), nq=int(_log(rng, 1, 10_000)),
                 side_lo=_log(rng, 1e-4, 1e-2), side_hi=_log(rng, 1e-2, 1e-1))
        npoints = c["ntraj"] * _mean_length(c)
        c["nq"] = max(1, min(c["nq"], int(MAX_PAIRS / (npoints * _mean_area(c)))))
        c["want"] = "pairs" if _most_pairs(c) < 60_000 else "digests"
        return c
    if op == "bitmap":
        c = {"op": op, "index": rng.choice(["grid", "stig", "fsg"]), **_database(rng, 10_000, 60_000)}
        c.update(cell=_cell(rng, c["ntraj"]), leaf=256, nq=int(_log(rng, 1, 300)), side_lo=_log(rng, 1e-3, 1e-2))
        c["side_hi"] = c["side_lo"] * rng.choice([1.0, 3.0])
        return c
    if op == "mixed":
        c = {"op": op, **_database(rng, 50_000, 300_000)}
        c.update(cell=rng.choice([0.002, 0.001]), leaf=256, nq=rng.randint(1_500, 9_000), side_lo=1e-4,
                 side_hi=_log(rng, 2e-2, 1e-1), group=rng.choice([1024, 2048]))
        return c
    if op == "topk":
        c = {"op": op, **_database(rng, 20_000, 200_000)}
        lo = rng.randint(8, 200)
        c.update(cell=_cell(rng, c["ntraj"]), nq=int(_log(rng, 1, 1000)), qlen_lo=lo,
                 qlen_hi=rng.randint(lo, 1024), k=int(_log(rng, 1, 100)))
        return c
    if op == "edr_all":
        c = {"op": op, **_database(rng, 2_000, 60_000)}
        lo = rng.randint(8, 300)
        c.update(cell=_cell(rng, c["ntraj"]), nq=rng.randint(1, 6), qlen_lo=lo, qlen_hi=rng.randint(lo, 1024))
        per_query = c["ntraj"] * _mean_length(c) * (c["qlen_lo"] + c["qlen_hi"]) / 2
        c["nq"] = max(1, min(c["nq"], int(MAX_CELLS / per_query)))
        return c
    if op == "similarity":
        c = {"op": op, **_database(rng, 5_000, 30_000)}
        lo = rng.randint(16, 200)
        c.update(cell=_cell(rng, c["ntraj"]), nq=rng.randint(1, 3), qlen_lo=lo, qlen_hi=lo + rng.randint(0, 200),
                 k=rng.randint(1, 50))
        return c
    c = {"op": op, "index": rng.choice(["grid", "mgrid", "fsg", "stig"]), **_database(rng, 5_000, 50_000)}
    c.update(cell=_cell(rng, c["ntraj"]), leaf=256)
    return c


def _trajectories(case: dict, seed: int) -> G.TrajSet:
    # The lengths belong to the case, so that a case has one size; the walks come from the seed.
    n = case["ntraj"]
    if case["lengths"] == "uniform":
        lengths = G.synth_lengths(n, n, "uniform", 16, 256, 16, 256)
    else:
        lengths = G.synth_lengths(n, n, "lognormal", case["median"], SIGMA, 8, 2048)
    return G.synth_walks(seed, lengths)


def _rects(case: dict, seed: int, hot: bool = False) -> np.ndarray:
    log_uniform = case["side_hi"] > case["side_lo"]
    if hot:
        return G.synth_rects(seed, case["nq"], case["side_lo"], case["side_hi"], log_uniform, 0.7, 16, 0.02)
    return G.synth_rects(seed, case["nq"], case["side_lo"], case["side_hi"], log_uniform)


def _queries(case: dict, seed: int, db: G.TrajSet) -> G.TrajSet:
    # The longest query length is always among them: it sets a batch's end.
    lengths = G.synth_lengths(seed + 1, case["nq"], "uniform", case["qlen_lo"], case["qlen_hi"], case["qlen_lo"],
                              case["qlen_hi"])
    lengths[-1] = case["qlen_hi"]
    # Every other query follows an indexed trajectory; a lone one does.
    return G.synth_queries(seed + 2, lengths, db, copy_mode=1 if case["nq"] == 1 else 2)


def _new_index(case: dict, kind: str):
    if kind == "stig":
        return G.StigIndex(case["leaf"])
    if kind == "fsg":
        return G.FsgIndex(UNIT_BOX, case["cell"])
    cls = G.MortonGridIndex if kind == "mgrid" else G.GridIndex
    return cls(UNIT_BOX, case["cell"], case.get("leaf", 256))


def prepare(case: dict, seed: int) -> dict:
    G.init(0)
    op = case["op"]
    db = _trajectories(case, seed)
    if op == "build":
        return {"case": case, "db": db}
    if op in ("range", "bitmap"):
        return {"case": case, "index": _new_index(case, case["index"]).build(db, device=True),
                "boxes": _rects(case, seed), "room": 8192 + 4 * _most_pairs(case)}
    if op == "mixed":
        parts = [_new_index(case, k).build(db, device=True) for k in ("grid", "stig", "fsg")]
        return {"case": case, "mixed": G.MixedRange(*parts), "boxes": _rects(case, seed, hot=True)}
    index = _new_index(case, "grid").build(db, device=True)
    return {"case": case, "index": index, "queries": _queries(case, seed, db)}


def _sorted_pairs(res, room: int) -> tuple[np.ndarray, np.ndarray]:
    """Per-query counts and every (query, trajectory, point) as one ascending
    64-bit key per hit (trajectory ids below 2^24, point ids below 2^16), in a
    table of `room` keys, unused ones -1; more hits than that are an error."""
    counts = res.counts()
    pairs = res.pairs()
    key = np.repeat(np.arange(len(counts), dtype=np.int64) << 40, counts)
    key |= (pairs[:, 0].astype(np.int64) << 16) | pairs[:, 1]
    key.sort()
    table = np.full(room, -1, np.int64)
    table[:len(key)] = key
    return counts, table


def run(state: dict):
    case = state["case"]
    op = case["op"]
    if op == "range":
        res = state["index"].range_batched(state["boxes"], graph=case["nq"] > 256)
        if case["want"] == "pairs":
            return _sorted_pairs(res, state["room"])
        return res.counts(), res.digests().view(np.int64)
    if op == "bitmap":
        return state["index"].range_bitmap(state["boxes"])
    if op == "mixed":
        counts, digests, route, _ = state["mixed"].run(state["boxes"], group_size=case["group"])
        return counts.astype(np.int64), digests.view(np.int64), route
    if op == "topk":
        ids, dists, _ = state["index"].similarity_batched(state["queries"], case["k"], EPS)
        return ids, dists
    if op == "edr_all":
        return state["index"].edr_batched_all(state["queries"], EPS)[0]
    if op == "similarity":
        return state["index"].similarity(state["queries"], case["k"], EPS)
    index = _new_index(case, case["index"]).build(state["db"], device=True)
    xy, ids, _, _ = index.fetch_store()
    if case["index"] != "stig":
        return xy, ids.view(np.int32), index.cell_starts()
    nodes = index.tree_nodes()[0]  # the shape of the kd-tree follows from the point count alone
    return xy, ids.view(np.int32), nodes["box"], nodes["start"].astype(np.int64), nodes["count"].astype(np.int64)


def work(case: dict) -> dict:
    op = case["op"]
    npoints = case["ntraj"] * _mean_length(case)
    if op == "build":
        # Coordinates up, the store (12 B a point) written and read back.
        return {"bytes": npoints * (8 + 12 + 12), "flops": 0}
    if op in ("range", "bitmap", "mixed"):
        pairs = case["nq"] * npoints * _mean_area(case)
        read = 12 * min(pairs, npoints)  # a point of several rectangles is read once
        if op == "bitmap":
            return {"bytes": read + 2 * case["nq"] * (case["ntraj"] + 1), "flops": 0}
        # Pairs written, and read by their consumer.
        return {"bytes": read + 16 * pairs + 32 * case["nq"], "flops": 0}
    qlen = (case["qlen_lo"] + case["qlen_hi"]) / 2
    if op == "topk":
        # The copied trajectory of every other query and about eight overlapping ones.
        cells = case["nq"] * (0.5 * qlen * qlen + 8 * qlen * _mean_length(case))
        return {"bytes": case["nq"] * (16 * qlen + 8 * case["k"]) + 16 * cells / qlen, "flops": 10 * cells}
    cells = case["nq"] * qlen * npoints
    out = 8 * case["nq"] * case["k"] if op == "similarity" else 4 * case["nq"] * case["ntraj"]
    return {"bytes": 8 * npoints + out, "flops": 10 * cells}


def tolerance(case: dict):
    return "exact"
