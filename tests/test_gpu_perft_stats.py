"""The statistics of a single position's perft, which runs stream-ordered, are
those of the level driver: one expand launch per level, and the arena its
levels take."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [1, 2, 3, 4, 6])
def test_perft_statistics(pg, depth):
    pos = pg.fen_to_pos("r3k2r/p1ppqpb1/bn2pnp1/3PN3/1p2P3/2N2Q1p/PPPBBPPP/R3K2R w KQkq - 0 1")
    eng = pg.Engine(backend="ks", arena_bytes=4 << 30)
    try:
        got = []
        for call in (lambda: eng.perft(pos, depth),
                     lambda: int(eng.perft_batch([pos], depth, mode=pg.MODE_LEVELS)[0])):
            eng.reset_stats()
            n = call()
            st = eng.stats()
            got.append((n, st["levels_run"], st["last_expand_launches"], st["peak_arena_bytes"], st["chunks"]))
            assert (st["last_expand_ms"] > 0) == (depth > 1)
            assert st["last_expand_ms"] * st["last_expand_launches"] <= st["gpu_ms"] * 1.001
        assert got[0] == got[1]
    finally:
        eng.close()
