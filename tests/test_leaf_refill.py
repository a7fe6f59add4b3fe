"""Waves whose 64 parents hand out more records than their list holds (640,
perft_gpu_amd/csrc/leaf_dev.h): the rest of the wave's calls are done in a
second round.  Through every kernel with a leaf pass by sets; the counts to
reach are those of one position at a time, whose levels run move by move."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "refill_check.cpp")
LIB = os.path.join(HERE, "native", "_build", "librefill_check.so")
CSRC = os.path.join(HERE, "..", "perft_gpu_amd", "csrc")
POOL = 640  # records a wave's list holds


@pytest.fixture(scope="module")
def rc():
    deps = [SRC] + [os.path.join(CSRC, f) for f in ("board.h", "sliders.h", "movegen.h", "leaf.h", "convert.h")]
    if not (os.path.exists(LIB) and all(os.path.getmtime(LIB) >= os.path.getmtime(d) for d in deps)):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        subprocess.run(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip", SRC, "-o", LIB],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    lib = ctypes.CDLL(LIB)
    lib.rc_records.argtypes = [ctypes.c_void_p]
    lib.rc_below.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return lib


@pytest.fixture(scope="module")
def positions(pg, rc):
    """48 positions of whose leaf parents at perft 4 (two plies below) 64 hand
    out more records than a list holds, on average"""
    base = pg.playouts(500, 20000, 20, 50, min_moves=40, no_check=True)
    rec = np.array([rc.rc_records(base[i:].ctypes.data) for i in range(len(base))])
    base = base[np.argsort(-rec)[:400]]
    n, mean, parents = ctypes.c_int(), [], []
    for i in range(len(base)):
        below = rc.rc_below(base[i:].ctypes.data, ctypes.byref(n))
        mean.append(below / max(n.value, 1))
        parents.append(n.value)
    best = np.argsort(-np.array(mean))[:48]
    return base[best], np.array(mean)[best], np.array(parents)[best]


def test_positions_overfill_a_list(positions):
    _, mean, parents = positions
    assert mean.min() * 64 > POOL
    assert parents.sum() > 768 * 64  # a whole wave of parents for every workgroup


@pytest.fixture(scope="module")
def want(pg, engine, positions, oracle):
    pos = positions[0]
    n = np.array([engine.perft(pg.Pos48(*[int(x) for x in p]), 4) for p in pos], dtype=np.uint64)
    assert np.array_equal(n[:6], oracle.perft_batch(pos[:6], 4, nthreads=8))
    return n


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
def test_table_free(pg, engine, positions, want, backend):
    engine.set_backend(backend)
    try:
        for mode in (pg.MODE_STREAM, pg.MODE_LEVELS, pg.MODE_PERSISTENT):
            assert np.array_equal(engine.perft_batch(positions[0], 4, mode=mode), want), mode
    finally:
        engine.set_backend("ks")


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
def test_table(pg, positions, want, backend):
    """the last write level with its leaf pass in one launch, two launches, and
    level by level from the host: the same counts and the same children made"""
    made = []
    for graphs, dedup in ((True, False), (False, False), (True, True)):
        eng = pg.Engine(backend=backend, arena_bytes=8 << 30, tt_bytes=1 << 28, zobrist_seed=7)
        try:
            eng.set_level_graphs(graphs)
            eng.set_dedup(dedup)
            eng.reset_stats()
            assert np.array_equal(eng.perft_batch(positions[0], 4), want), (graphs, dedup)
            if not dedup:  # (which child claims a slot, and so which finds none, differs from run to run)
                made.append(eng.stats()["made_nodes"])
        finally:
            eng.close()
    assert made[0] == made[1]


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
@pytest.mark.parametrize("tt_bytes", [0, 1 << 28])
def test_serving(pg, positions, want, backend, tt_bytes):
    pos = positions[0]
    eng = pg.Engine(backend=backend, arena_bytes=8 << 30, tt_bytes=tt_bytes)
    try:
        eng.serve_start(max_jobs=64)
        for i in range(len(pos)):
            eng.submit(pos[i], 4, i)
        got = {}
        while len(got) < len(pos):
            got.update((r["tag"], (r["status"], r["nodes"])) for r in eng.poll())
        eng.serve_stop()
        assert got == {i: (0, int(w)) for i, w in enumerate(want)}
    finally:
        eng.close()
