"""The leaf level by sets (perft_gpu_amd/csrc/leaf.h): perft 2 summed per set
of moves equals perft 2 move by move, on the CPU over played and over randomly
placed positions, and on the GPU at the sizes where its tiles, record lists
and dispatch have their edges."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "leaf_check.cpp")
LIB = os.path.join(HERE, "native", "_build", "libleaf_check.so")
CSRC = os.path.join(HERE, "..", "perft_gpu_amd", "csrc")

SPECIAL = [
    "rnbqkbnr/pppppppp/8/8/8/8/PPPPPPPP/RNBQKBNR w KQkq - 0 1",
    "r3k2r/p1ppqpb1/bn2pnp1/3PN3/1p2P3/2N2Q1p/PPPBBPPP/R3K2R w KQkq - 0 1",
    "8/2p5/3p4/KP5r/1R3p1k/8/4P1P1/8 w - - 0 1",
    "r3k2r/Pppp1ppp/1b3nbN/nP6/BBP1P3/q4N2/Pp1P2PP/R2Q1RK1 w kq - 0 1",
    "rnbq1k1r/pp1Pbppp/2p5/8/2B5/8/PPP1NnPP/RNBQK2R w KQ - 1 8",
    "3Q4/1Q4Q1/4Q3/2Q4R/Q4Q2/3Q4/1Q4Rp/1K1BBNNk w - - 0 1",
    "r3k2r/8/3Q4/8/8/5q2/8/R3K2R b KQkq - 0 1",
    "8/8/8/8/k2Pp2Q/8/8/3K4 b - d3 0 1",
    "4k3/4r3/8/8/4P3/8/4P3/4K3 w - - 0 1",
    "8/1p1p1p2/8/P1P1P1P1/8/8/8/K6k w - - 0 1",
    "2r5/3pk3/8/2P5/8/2K5/8/8 w - - 0 1",
    "8/8/1k6/2b5/2pP4/8/5K2/8 b - d3 0 1",
]


@pytest.fixture(scope="module")
def leaf():
    deps = [SRC] + [os.path.join(CSRC, f) for f in ("board.h", "sliders.h", "movegen.h", "leaf.h", "convert.h")]
    if not (os.path.exists(LIB) and all(os.path.getmtime(LIB) >= os.path.getmtime(d) for d in deps)):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        subprocess.run(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip", SRC, "-o", LIB],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    lib = ctypes.CDLL(LIB)
    lib.lc_perft2.restype = lib.lc_perft2_moves.restype = ctypes.c_uint64
    lib.lc_perft2.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    lib.lc_perft2_moves.argtypes = [ctypes.c_void_p]
    lib.lc_unsound.argtypes = [ctypes.c_void_p]
    lib.lc_random.argtypes = [ctypes.c_uint64, ctypes.c_int, ctypes.c_void_p]
    return lib


def _random(pg, leaf, seed, n):
    pos = np.zeros(n, dtype=pg.POS_DTYPE)
    leaf.lc_random(seed, n, pos.ctypes.data)
    return pos


def _records(leaf, pos):
    st, out = (ctypes.c_int * 4)(), []
    for i in range(len(pos)):
        leaf.lc_perft2(pos[i:].ctypes.data, st)
        out.append(st[0])
    return np.array(out)


@pytest.mark.parametrize("plies", [(1, 8), (8, 40), (40, 120), None])
def test_sets_equal_moves(pg, leaf, plies):
    pos = pg.playouts(31 + plies[0], 6000, *plies) if plies else _random(pg, leaf, 5, 20000)
    st = (ctypes.c_int * 4)()
    by_set = 0
    for i in range(len(pos)):
        p = pos[i:].ctypes.data
        got, want = leaf.lc_perft2(p, st), leaf.lc_perft2_moves(p)
        assert got == want, pos[i]
        assert st[3] == 0
        by_set += st[2] == 0
    assert by_set  # some positions need no child counted in full


def test_sets_equal_oracle(pg, leaf, oracle):
    for fen in SPECIAL:
        p = pg.fen_to_pos(fen)
        arr = pg.positions_array([p])
        assert leaf.lc_perft2(arr.ctypes.data, None) == oracle.perft_fen(fen, 2), fen
    pos = pg.playouts(77, 400, 6, 60)
    want = oracle.perft_batch(pos, 2, nthreads=8)
    assert [leaf.lc_perft2(pos[i:].ctypes.data, None) for i in range(len(pos))] == [int(x) for x in want]


# roots of a depth-2 batch are leaf parents themselves: below 32 a workgroup
# (768 workgroups) they run move by move, from there by sets, in tiles of up
# to 256
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 24575, 24576, 24577, 50021, 196608, 196609])
def test_leaf_level_sizes(pg, oracle, engine, n):
    base = np.concatenate([pg.playouts(9, 700, 6, 60), pg.positions_array([pg.fen_to_pos(f) for f in SPECIAL])])
    want = oracle.perft_batch(base, 2, nthreads=8).astype(np.int64)
    at = np.arange(n) % len(base)
    for mode in (pg.MODE_STREAM, pg.MODE_LEVELS, pg.MODE_PERSISTENT):
        got = engine.perft_batch(np.ascontiguousarray(base[at]), 2, mode=mode)
        assert np.array_equal(got.astype(np.int64), want[at]), mode


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
def test_leaf_level_roots_mixed(pg, oracle, engine, backend):
    """leaf tiles that hold parents of several roots, at levels on either side
    of the dispatch's line"""
    pos = pg.playouts(1234, 150, 8, 60)
    engine.set_backend(backend)
    try:
        for n, d in ((3, 3), (150, 3), (20, 4), (40, 4), (150, 4)):
            want = oracle.perft_batch(pos[:n], d, nthreads=8)
            for mode in (pg.MODE_STREAM, pg.MODE_LEVELS):
                assert np.array_equal(engine.perft_batch(pos[:n], d, mode=mode), want), (n, d, mode)
    finally:
        engine.set_backend("ks")


@pytest.mark.gpu
def test_leaf_records_overflow(pg, leaf, engine):
    """waves whose parents hand out more records than their list holds (640 for
    64 parents) and tiles with many move windows: the positions with the most
    records and the most moves to make, of random placements"""
    pos = _random(pg, leaf, 8, 40000)
    rec = _records(leaf, pos)
    many = pos[np.argsort(-rec)[:128]]
    assert _records(leaf, many).min() > 10
    for base in (many, pos[:2000]):
        # a batch this small runs move by move
        want = engine.perft_batch(np.ascontiguousarray(base), 2, mode=pg.MODE_STREAM)
        at = np.arange(30011) % len(base)
        got = engine.perft_batch(np.ascontiguousarray(base[at]), 2, mode=pg.MODE_STREAM)
        assert np.array_equal(got, want[at])
        # (elsewhere only the GPU's own paths can be compared)
        sound = [i for i in range(len(base)) if not leaf.lc_unsound(base[i:].ctypes.data)]
        assert sound
        for i in sound:
            assert int(got[i]) == leaf.lc_perft2_moves(base[i:].ctypes.data), base[i]


@pytest.mark.gpu
@pytest.mark.parametrize("backend,graphs,dedup", [("ks", True, True), ("ks", False, True), ("ks", False, False),
                                                  ("fancy", True, True), ("byte", False, True)])
def test_table_leaf_level(pg, oracle, backend, graphs, dedup):
    """leaf passes of the table search on either side of 32 parents a
    workgroup, in planned passes (two launches, or the last write level and
    its leaf pass in one) and level by level from the host"""
    pos = pg.playouts(4321, 1500, 8, 60)
    for n, d in ((1, 3), (40, 3), (701, 3), (20, 4), (900, 4), (1500, 4), (60, 5)):
        want = oracle.perft_batch(pos[:n], d, nthreads=8)
        eng = pg.Engine(backend=backend, arena_bytes=4 << 30, tt_bytes=1 << 28, zobrist_seed=7)
        try:
            eng.set_level_graphs(graphs)
            eng.set_dedup(dedup)
            assert np.array_equal(eng.perft_batch(pos[:n], d), want), (n, d)
        finally:
            eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("tt_bytes", [0, 1 << 28])
@pytest.mark.parametrize("jobs,n,dmax", [(1, 6, 4), (4, 30, 4), (64, 300, 4), (64, 200, 5)])
def test_serving_step_forms(pg, oracle, tt_bytes, jobs, n, dmax):
    """steps small enough for the fewer launches, finely tiled ones and large
    ones, with leaf passes in the write's step and after it"""
    pos = pg.playouts(99, n, 8, 60)
    depth = [1 + (i * 7) % dmax for i in range(n)]
    want = {}
    for d in sorted(set(depth)):
        sel = [i for i in range(n) if depth[i] == d]
        want.update(zip(sel, oracle.perft_batch(np.ascontiguousarray(pos[sel]), d, nthreads=8)))
    eng = pg.Engine(arena_bytes=4 << 30, tt_bytes=tt_bytes)
    try:
        for wait_each in (True, False):
            eng.serve_start(max_jobs=jobs)
            got = {}
            for i in range(n):
                eng.submit(pos[i], depth[i], i)
                while wait_each and i not in got:
                    got.update((r["tag"], r["nodes"]) for r in eng.poll())
            while len(got) < n:
                got.update((r["tag"], r["nodes"]) for r in eng.poll())
            eng.serve_stop()
            assert got == {i: int(w) for i, w in want.items()}
    finally:
        eng.close()


@pytest.mark.gpu
def test_table_leaf_made_nodes(pg):
    """the write level that runs with its leaf pass leaves its children's moves
    to that pass: the same counts and the same number of children made as level
    by level, where the write counts them"""
    pos = pg.playouts(2024, 40, 15, 50, min_moves=35, no_check=True)
    got = []
    for graphs in (True, False):
        eng = pg.Engine(arena_bytes=48 << 30, tt_bytes=1 << 30, zobrist_seed=3)
        try:
            eng.set_level_graphs(graphs)
            eng.set_dedup(False)  # (which child claims a slot, and so which finds none, differs from run to run)
            eng.reset_stats()
            n = eng.perft_batch(pos, 6)
            st = eng.stats()
            got.append(([int(x) for x in n], st["made_nodes"], st["frontier_nodes"]))
            assert (st["graph_passes"] > 0) == graphs
        finally:
            eng.close()
    assert got[0] == got[1]
