"""Stream-ordered batches of at most 1024 roots, whose begin and outcome are
one launch each: on either side of the sizes of a wave and of the workgroup,
from host and device buffers, alone and from several threads, and where a
level does not fit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pos(pg, p):
    return pg.Pos48(*[int(x) for x in p])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025])
@pytest.mark.parametrize("backend", ["ks", "byte"])
def test_sizes(pg, oracle, engine, n, backend):
    pos = pg.playouts(6, n, 2, 70)
    engine.set_backend(backend)
    try:
        for d in (1, 2, 3):
            want = oracle.perft_batch(pos, d, nthreads=8)
            assert np.array_equal(engine.perft_batch(pos, d, mode=pg.MODE_STREAM), want), d
            din, dout = pg.DeviceArray.from_host(pos), pg.DeviceArray(n, np.uint64)
            engine.perft_batch_ptr(din.ptr, n, d, dout.ptr, pg.MODE_STREAM)
            assert np.array_equal(dout.download(), want), d
            dout.upload(np.full(n, 77, dtype=np.uint64))
            engine.perft_batch_noalloc_ptr(din.ptr, n, d, dout.ptr)
            assert np.array_equal(dout.download(), want), d
            assert engine.perft(_pos(pg, pos[0]), d) == int(want[0])
    finally:
        engine.set_backend("ks")


def test_level_that_does_not_fit(pg, oracle):
    """one position runs stream-ordered, or in chunks where a level is larger
    than the arena; a refused batch leaves the context usable"""
    start = pg.fen_to_pos(pg.START_FEN)
    pos = pg.playouts(8, 40, 8, 60)
    eng = pg.Engine(arena_bytes=1 << 20)
    try:
        for _ in range(2):
            assert eng.perft(start, 5) == 4865609
            eng.reset_stats()
            assert eng.perft(start, 6) == 119060324
            assert eng.stats()["chunks"] > 0
            with pytest.raises(pg.PerftError):
                eng.perft_batch(pos, 4, mode=pg.MODE_STREAM)
            assert np.array_equal(eng.perft_batch(pos, 4), oracle.perft_batch(pos, 4, nthreads=8))
            assert eng.perft(start, 3) == 8902
    finally:
        eng.close()


def test_contexts_on_threads(pg, oracle):
    """two contexts, each with its own outcome words, from two threads at once"""
    pos = pg.playouts(13, 200, 4, 60)
    want = {d: oracle.perft_batch(pos, d, nthreads=8) for d in (1, 2, 3)}
    bad = []

    def work(k):
        eng = pg.Engine(arena_bytes=1 << 28)
        try:
            for i in range(60):
                d = 1 + (i + k) % 3
                n = 1 + (i * 37 + k) % 200
                if not np.array_equal(eng.perft_batch(pos[:n], d), want[d][:n]):
                    bad.append((k, i))
                if eng.perft(_pos(pg, pos[i]), d) != int(want[d][i]):
                    bad.append((k, i, "one"))
        finally:
            eng.close()

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
def test_parents_per_tile(pg, oracle, engine, backend):
    """tiles of 4, 5, 8 and 9 parents (768 workgroups), whose moves are
    generated by 64 and by 32 threads a parent and by one"""
    pos = pg.playouts(21, 500, 2, 90)
    want = oracle.perft_batch(pos, 2, nthreads=8)
    engine.set_backend(backend)
    try:
        for n in (3071, 3072, 3073, 6143, 6144, 6145):
            at = np.arange(n) % len(pos)
            for mode in (pg.MODE_STREAM, pg.MODE_LEVELS):
                got = engine.perft_batch(np.ascontiguousarray(pos[at]), 2, mode=mode)
                assert np.array_equal(got, want[at]), (n, mode)
    finally:
        engine.set_backend("ks")
