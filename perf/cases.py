"""Timing cases of the perft engine: the calls a program makes, over the range
of sizes it makes them with.

A case names a call (`kind`), its depth, its number of positions, the slider
backend, how the positions were played (`plies`: random legal playouts of at
most that many plies, as the engine's own workloads use) and, for runs with a
transposition table, the table's size.  Every call returns its exact counts.
"""
import math
import weakref

import numpy as np
import torch

import perft_gpu_amd as pg
from perft_gpu_amd.workloads import C2_OPS_PER_LEAF, C4

GIB = 1 << 30

# Moves per position that expected sizes are reckoned with (random playouts of
# 8 to 60 plies average 30 to 33).
BRANCH = 31.0

BACKENDS = ("ks", "plain", "fancy", "byte")


def listed():
    return [
        # one position, a shallow count: latency of the plain call
        dict(name="one-d3", kind="one", depth=3, n=1, backend="ks", plies=20),
        # one position at the depth of a quick move-generator check
        dict(name="one-d5", kind="one", depth=5, n=1, backend="ks", plies=30),
        # one position, deep enough to fill the device, plain magics
        dict(name="one-d6-plain", kind="one", depth=6, n=1, backend="plain", plies=40),
        # UCI "go perft 5": the counts of every root move
        dict(name="divide-d5", kind="divide", depth=5, n=1, backend="ks", plies=24),
        # a small ragged batch from host memory, byte-lookup tables
        dict(name="batch-37-d4-byte", kind="batch", depth=4, n=37, backend="byte", plies=40),
        # a batch on device buffers for callers that may not allocate
        dict(name="noalloc-100-d4", kind="noalloc", depth=4, n=100, backend="ks", plies=40),
        # the benchmark's batch: 256 positions at depth 5, resident in HBM
        dict(name="batch-256-d5", kind="device", depth=5, n=256, backend="ks", plies=40),
        # a larger ragged batch from host memory, the reference's default backend
        dict(name="batch-701-d5-fancy", kind="batch", depth=5, n=701, backend="fancy", plies=50),
        # serving, one request at a time: latency of a running server
        dict(name="serve-one-d4", kind="serve", depth=4, n=1, backend="ks", plies=60, table_gib=0),
        # serving, a burst with the request mix of the serving workload (depths
        # 3 to 7), from start to drained, on an emptied shared table
        dict(name="serve-burst-200", kind="burst", depth=7, n=200, backend="ks", plies=60, table_gib=8),
        # one middlegame position at depth 8 with an emptied table
        dict(name="table-one-d8", kind="table", depth=8, n=1, backend="ks", plies=30, table_gib=16),
        # high-mobility positions at depth 6 sharing an emptied table
        dict(name="table-batch-256-d6", kind="table", depth=6, n=256, backend="ks", plies=50, table_gib=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("one", "divide", "batch", "batch", "device", "device", "noalloc", "serve", "burst", "table"))
    case = dict(kind=kind, backend=rng.choice(BACKENDS), plies=rng.randint(12, 60), n=1)
    if kind in ("one", "divide"):
        case["depth"] = rng.randint(2, 6)
    elif kind in ("batch", "device"):
        case["depth"] = rng.randint(2, 5)
        case["n"] = _log_int(rng, 1, 1000 if case["depth"] == 5 else 8000)
    elif kind == "noalloc":
        case["depth"] = rng.randint(2, 5)
        case["n"] = _log_int(rng, 1, 96 if case["depth"] == 5 else 2000)
    elif kind == "serve":
        case["depth"] = rng.randint(2, 5)
        case["n"] = _log_int(rng, 1, 12)
        case["table_gib"] = 0
    elif kind == "burst":
        case["depth"] = rng.randint(4, 7)
        case["n"] = _log_int(rng, 20, 200)
        case["table_gib"] = rng.choice((1, 2, 4, 8))
    elif rng.random() < 0.5:
        case["depth"] = rng.randint(5, 7)
        case["table_gib"] = rng.choice((1, 4, 16))
    else:
        case["depth"] = rng.randint(4, 6)
        case["n"] = _log_int(rng, 3, 250)
        case["table_gib"] = rng.choice((2, 8, 16))
    return case


def _request_depths(case):
    """Depths of a burst's requests: the serving workload's shares, in order of
    a fixed shuffle, none deeper than the case's."""
    depths, n = [], case["n"]
    for d, p in zip(C4["depths"], C4["probs"]):
        depths += [min(d, case["depth"])] * max(1, round(p * n))
    depths = (depths + [3] * n)[:n]
    order = np.random.RandomState(7).permutation(n)
    return [depths[i] for i in order]


class _Holder:
    """An engine and, for the serving cases, its running server: a program
    keeps one and sends it every input."""

    def __init__(self, backend, table_gib, arena, serving):
        self.engine = pg.Engine(backend=backend, arena_bytes=arena, tt_bytes=table_gib * GIB, zobrist_seed=7)
        if serving:
            self.engine.serve_start(max_jobs=64)

    def __del__(self):
        if hasattr(self, "engine"):
            self.engine.close()


_holders = weakref.WeakValueDictionary()


def _holder(case):
    table = case.get("table_gib", 0)
    key = (case["backend"], table, 24 * GIB if case["kind"] == "table" else 16 * GIB, case["kind"] == "serve")
    h = _holders.get(key)
    if h is None:
        h = _holders[key] = _Holder(*key)
    return h


def prepare(case, seed):
    kind, n, plies = case["kind"], case["n"], case["plies"]
    # high-mobility positions where a table is used, any otherwise
    min_moves = 35 if kind == "table" else 0
    pos = pg.playouts(seed * 2654435761 % (1 << 62) + 1, n, max(8, plies // 2) if kind != "one" else plies, plies,
                      min_moves, kind == "table")
    h = _holder(case)
    state = dict(kind=kind, depth=case["depth"], n=n, holder=h, engine=h.engine, pos=pos)
    if kind in ("one", "serve", "burst", "divide"):
        state["list"] = [pg.Pos48(*[int(x) for x in p]) for p in pos]
    if kind in ("device", "noalloc"):
        state["dpos"] = torch.from_numpy(pos.view(np.int64).reshape(n, 6)).cuda()
        state["dout"] = torch.zeros(n, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
    if kind == "serve":
        state["depths"] = [case["depth"]] * n
    if kind == "burst":
        state["depths"] = _request_depths(case)
    return state


def _collect(engine, requests, depths):
    """Submit every request, then poll until each is answered."""
    for tag, (pos, depth) in enumerate(zip(requests, depths)):
        engine.submit(pos, depth, tag)
    out = np.zeros(len(requests), dtype=np.int64)
    left = len(requests)
    while left:
        for r in engine.poll(256):
            if r["status"]:
                raise RuntimeError("request %d: status %d" % (r["tag"], r["status"]))
            out[r["tag"]] = r["nodes"]
            left -= 1
    return out


def run(state):
    eng, kind, depth = state["engine"], state["kind"], state["depth"]
    if kind == "one":
        return eng.perft(state["list"][0], depth)
    if kind == "divide":
        counts = np.zeros(256, dtype=np.int64)  # a position has at most 218 moves
        for i, (_, c) in enumerate(eng.divide(state["list"][0], depth)):
            counts[i] = c
        return counts
    if kind == "batch":
        return eng.perft_batch(state["pos"], depth).astype(np.int64)
    if kind == "device":
        eng.perft_batch_ptr(state["dpos"].data_ptr(), state["n"], depth, state["dout"].data_ptr())
        return state["dout"]
    if kind == "noalloc":
        eng.perft_batch_noalloc_ptr(state["dpos"].data_ptr(), state["n"], depth, state["dout"].data_ptr())
        return state["dout"]
    if kind == "serve":
        return _collect(eng, state["list"], state["depths"])
    # with a table: on an emptied one, so that every pass computes its counts
    eng.set_tt_regions(0)
    if kind == "burst":
        eng.serve_start(max_jobs=256)
        try:
            return _collect(eng, state["list"], state["depths"])
        finally:
            eng.serve_stop()
    return eng.perft_batch(state["pos"], depth).astype(np.int64)


def work(case):
    """Positions in, counts out, and the integer operations of the counting:
    the benchmark's operations per leaf times the expected leaves.  With a
    table, each ply below the fourth finds some 40% of its positions to be
    transpositions."""
    kind, n, depth = case["kind"], case["n"], case["depth"]
    if kind == "burst":
        leaves = sum(BRANCH ** d * 0.6 ** max(0, d - 4) for d in _request_depths(case))
    else:
        leaves = n * BRANCH ** depth
        if kind == "table":
            leaves *= 0.6 ** max(0, depth - 4)
    outs = 8 * (BRANCH if kind == "divide" else n)
    return {"bytes": 48 * n + outs, "flops": C2_OPS_PER_LEAF * leaves}


def exact(case, seed):
    """Counts are whole numbers, equal or wrong: nothing here is rounded."""
    return None
