"""Positions that are no chess: raw positions on which a side has no king or
several (the FEN parser refuses them, the calls take them).  Their counts
follow the move generator's conventions and must not depend on the form in
which a level runs."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "kings_check.cpp")
LIB = os.path.join(HERE, "native", "_build", "libkings_check.so")
CSRC = os.path.join(HERE, "..", "perft_gpu_amd", "csrc")


@pytest.fixture(scope="module")
def kings():
    deps = [SRC] + [os.path.join(CSRC, f) for f in ("board.h", "sliders.h", "movegen.h", "leaf.h", "convert.h")]
    if not (os.path.exists(LIB) and all(os.path.getmtime(LIB) >= os.path.getmtime(d) for d in deps)):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        subprocess.run(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip", SRC, "-o", LIB],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    lib = ctypes.CDLL(LIB)
    lib.kc_disagree.argtypes = [ctypes.c_void_p, ctypes.c_int]
    return lib


def _random(pg, seed, n, white, black):
    """n random placements with that many kings a side (None: up to three)"""
    r = np.random.RandomState(seed)
    out = np.zeros(n, dtype=pg.POS_DTYPE)
    names = out.dtype.names
    for i in range(n):
        free = list(r.permutation(64))
        f = dict.fromkeys(("white_pieces", "pawns", "knights", "bishop_queens", "rook_queens", "kings"), 0)

        def put(field, side, ranks=range(8)):
            at = next((s for s in free if s >> 3 in ranks), None)
            if at is None:
                return
            free.remove(at)
            for name in field:
                f[name] |= 1 << int(at)
            if side:
                f["white_pieces"] |= 1 << int(at)

        for side, k in ((1, white), (0, black)):
            for _ in range(r.randint(0, 4) if k is None else k):
                put(["kings"], side)
        for field, most, ranks in ((["pawns"], 10, range(1, 7)), (["knights"], 4, range(8)),
                                   (["bishop_queens"], 4, range(8)), (["rook_queens"], 4, range(8)),
                                   (["bishop_queens", "rook_queens"], 3, range(8))):
            for _ in range(r.randint(0, most + 1)):
                put(field, r.randint(2), ranks)
        f["pawns"] |= int(r.randint(2)) << 63
        for name in names:
            out[name][i] = f[name]
    return out


@pytest.mark.parametrize("white,black", [(1, 1), (1, 2), (2, 1), (2, 2), (3, 3), (1, 0), (0, 1), (0, 0), (None, None)])
def test_forms_agree(pg, kings, white, black):
    pos = _random(pg, 3, 3000, white, black)
    bad = [(i, kings.kc_disagree(pos[i:].ctypes.data, i < 200)) for i in range(len(pos))]
    bad = [x for x in bad if x[1]]
    assert not bad, (len(bad), bad[:5])


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
def test_levels_agree(pg, engine, backend):
    """the same positions in tiles of four, sixteen and forty parents a
    workgroup (generated by the whole workgroup, by a lane each, and summed by
    sets)"""
    base = np.concatenate([_random(pg, 5, 150, w, b) for w, b in ((2, 2), (3, 1), (1, 0), (0, 1), (None, None))])
    engine.set_backend(backend)
    try:
        got = []
        for n in (len(base), 768 * 16, 768 * 40):
            at = np.arange(n) % len(base)
            got.append(engine.perft_batch(np.ascontiguousarray(base[at]), 2, mode=pg.MODE_STREAM))
            assert np.array_equal(got[-1], got[-1][:len(base)][at])
        assert np.array_equal(got[0], got[1][:len(base)]) and np.array_equal(got[0], got[2][:len(base)])
        deep = [engine.perft_batch(base[:300], 3, mode=m) for m in (pg.MODE_STREAM, pg.MODE_LEVELS)]
        assert np.array_equal(deep[0], deep[1])
        if backend != "ks":
            engine.set_backend("ks")
            assert np.array_equal(engine.perft_batch(base, 2), got[0])
    finally:
        engine.set_backend("ks")


def _bogus_rights(pg, seed, n):
    """one king a side, back ranks thinned out, every castling right set: the
    FEN parser takes rights whose king or rook is not at home, and a castle
    then puts a rook where another piece may stand"""
    pos = _random(pg, seed, n, 1, 1)
    for name in pos.dtype.names:
        if name not in ("kings", "white_pieces"):
            pos[name] &= np.uint64(~0x7E0000000000007E & (1 << 64) - 1)
    pos["pawns"] |= np.uint64(15)
    return pos


FENS = ["n6n/8/5P2/6K1/7R/2k5/5N2/8 b Qq - 0 1", "n4n2/5KRr/1bp3QP/3k3P/3p3p/3PQ2R/p2P3b/5Q2 b kq - 0 1",
        "8/3k4/8/2K5/8/8/p6p/N6B w KQ - 0 1", "4k2n/8/8/8/8/8/5P2/4K2N b KQkq - 0 1"]


def test_rights_without_rook(pg, kings):
    pos = np.concatenate([pg.positions_array([pg.fen_to_pos(f) for f in FENS]), _bogus_rights(pg, 21, 600)])
    bad = [(i, kings.kc_disagree(pos[i:].ctypes.data, 1)) for i in range(len(pos))]
    bad = [x for x in bad if x[1]]
    assert not bad, (len(bad), bad[:5])


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
def test_rights_without_rook_levels(pg, engine, backend):
    base = np.concatenate([pg.positions_array([pg.fen_to_pos(f) for f in FENS]), _bogus_rights(pg, 23, 60)])
    engine.set_backend(backend)
    try:
        small = engine.perft_batch(base, 3)  # some 2,000 leaf parents: move by move
        at = np.arange(4000) % len(base)
        large = engine.perft_batch(np.ascontiguousarray(base[at]), 3)
        assert np.array_equal(large, small[at])
    finally:
        engine.set_backend("ks")


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["ks", "fancy"])
def test_serving_several_kings(pg, engine, backend):
    """the serving thread sizes a request's levels with the host's own count"""
    pos = np.concatenate([_random(pg, 9, 30, w, b) for w, b in ((2, 2), (3, 1), (1, 0), (None, None))])
    engine.set_backend(backend)
    try:
        want = engine.perft_batch(pos, 3)
    finally:
        engine.set_backend("ks")
    eng = pg.Engine(backend=backend, arena_bytes=1 << 30)
    try:
        eng.serve_start(max_jobs=32)
        for i in range(len(pos)):
            eng.submit(pos[i], 3, i)
        got = {}
        while len(got) < len(pos):
            got.update((r["tag"], (r["status"], r["nodes"])) for r in eng.poll())
        eng.serve_stop()
        assert got == {i: (0, int(w)) for i, w in enumerate(want)}
    finally:
        eng.close()
