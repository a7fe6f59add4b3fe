"""A device buffer too small for a batch's counts is refused by
the small batches too, whose counts are written by a kernel where larger ones
are copied, and nothing is written."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 700, 1024])
def test_short_output_buffer(pg, oracle, engine, n):
    pos = pg.playouts(17, n, 4, 60)
    din, dout = pg.DeviceArray.from_host(pos), pg.DeviceArray(n - 1, np.uint64)
    dout.upload(np.full(n - 1, 77, dtype=np.uint64))
    with pytest.raises(pg.PerftError) as ei:
        engine.perft_batch_ptr(din.ptr, n, 2, dout.ptr, pg.MODE_STREAM)
    assert ei.value.status == pg.PF_EDEVICE
    assert (dout.download() == 77).all()
    # one that fits is written, at its end too
    want = oracle.perft_batch(pos, 2, nthreads=8)
    engine.perft_batch_ptr(din.ptr, n - 1, 2, dout.ptr, pg.MODE_STREAM)
    assert np.array_equal(dout.download(), want[:n - 1])
