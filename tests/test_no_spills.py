"""The kernels that hold a leaf tile (perft_gpu_amd/csrc/leaf_dev.h) keep every
vector register out of memory: the library's own kernel metadata says so.  The
leaf pass is the library's longest stretch of live values, 150 to 168 of the
168 vector registers that three waves per SIMD leave it; what does not fit goes
to scratch memory without a warning."""
import struct

import msgpack
import pytest

LEAF = ("k_stream_leaf", "k_expand_leaf", "k_persistent", "k_step_leaf", "k_step_write_leaf", "k_step_mixed",
        "k_step_late", "k_expand_tt_leaf")


@pytest.fixture(scope="module")
def kernels():
    """name -> metadata, from the AMDGPU notes of the code objects in the library"""
    from perft_gpu_amd import build
    data = open(build.LIB, "rb").read()
    found, at = {}, data.find(b"AMDGPU\0\0")
    while at >= 0:
        namesz, descsz, kind = struct.unpack_from("<III", data, at - 12)
        if (namesz, kind) == (7, 32):
            for k in msgpack.unpackb(data[at + 8:at + 8 + descsz])["amdhsa.kernels"]:
                found[k[".name"]] = k
        at = data.find(b"AMDGPU\0\0", at + 8)
    return found


@pytest.mark.parametrize("kernel", LEAF)
def test_leaf_kernels_do_not_spill(pg, kernels, kernel):
    mine = {n: k for n, k in kernels.items() if "%d%sI" % (len(kernel), kernel) in n}
    assert len(mine) >= 4  # one for each slider backend
    assert not {n: k[".vgpr_spill_count"] for n, k in mine.items() if k[".vgpr_spill_count"]}
