"""The stream-ordered write kernel has two forms; tune files that name one of the
five there were still load and count the same."""
import struct

import msgpack
import numpy as np
import pytest


def test_two_write_kernels_per_backend(pg):
    from perft_gpu_amd import build
    data = open(build.LIB, "rb").read()
    names, at = set(), data.find(b"AMDGPU\0\0")
    while at >= 0:
        namesz, descsz, kind = struct.unpack_from("<III", data, at - 12)
        if (namesz, kind) == (7, 32):
            names |= {k[".name"] for k in msgpack.unpackb(data[at + 8:at + 8 + descsz])["amdhsa.kernels"]}
        at = data.find(b"AMDGPU\0\0", at + 8)
    for b in range(4):
        assert sum("k_stream_writeILi%dE" % b in n for n in names) == 2


@pytest.mark.gpu
def test_files_with_older_forms(pg, oracle, tmp_path):
    pos = pg.playouts(31, 60, 8, 60)
    want = oracle.perft_batch(pos, 4, nthreads=8)
    path = tmp_path / "t.txt"
    for form in (-1, 0, 1, 2, 3, 4, 5, 6, 9):
        path.write_text("perft_gpu_amd tuning 1\nbackend ks stream_leaf 3 stream_write %d\n" % form)
        eng = pg.Engine(backend="ks", arena_bytes=1 << 30, tune_file=str(path))
        try:
            assert np.array_equal(eng.perft_batch(pos, 4, mode=pg.MODE_STREAM), want), form
            if form in (0, 4):
                eng.tune(pos, 3, str(tmp_path / "out.txt"))
                line = [s for s in open(tmp_path / "out.txt") if s.startswith("backend ks ")][0].split()
                assert line[line.index("stream_write") + 1] in ("0", "3")
        finally:
            eng.close()
