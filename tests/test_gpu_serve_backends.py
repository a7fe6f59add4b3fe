"""The serving step's kernels with every slider backend, in all forms of the
step: small ones (a request at a time), finely tiled ones (some tens) and
coarse ones (hundreds), on a server started more than once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def requests(pg, oracle):
    n = 260
    pos = pg.playouts(4242, n, 8, 60)
    depth = np.array([1 + (i * 7) % 5 for i in range(n)])
    want = np.zeros(n, dtype=np.int64)
    for d in range(1, 6):
        sel = np.nonzero(depth == d)[0]
        want[sel] = oracle.perft_batch(np.ascontiguousarray(pos[sel]), d, nthreads=8)
    return pos, depth, want


@pytest.mark.parametrize("backend", ["ks", "plain", "fancy", "byte"])
@pytest.mark.parametrize("tt_bytes", [0, 1 << 28])
def test_step_forms(pg, requests, backend, tt_bytes):
    pos, depth, want = requests
    eng = pg.Engine(backend=backend, arena_bytes=8 << 30, tt_bytes=tt_bytes, zobrist_seed=5)
    try:
        # (first, last, requests outstanding at a time)
        for first, last, window in ((0, 12, 1), (12, 60, 48), (0, 260, 260), (60, 72, 1)):
            eng.serve_start(max_jobs=256)
            got, sent = {}, first
            while len(got) < last - first:
                while sent < last and sent - first - len(got) < window:
                    eng.submit(pos[sent], int(depth[sent]), sent)
                    sent += 1
                got.update((r["tag"], (r["status"], r["nodes"])) for r in eng.poll())
            eng.serve_stop()
            assert got == {i: (0, int(want[i])) for i in range(first, last)}
    finally:
        eng.close()
