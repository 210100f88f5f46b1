"""Where the lanes of a buffer load read: numbers of the operand that the kernel wants, or nothing.  A lane that has nothing to read
is stopped by the range check with its own place alone, since a scalar place is not known to count in it.  The kernels' sums of
places are gone through on the host, with the functions that give the buffers; no GPU is needed."""
import ctypes
import re
import subprocess

import numpy as np
import pytest

from axon_amd.kernels import build as B

HOST = """#include "buffer.h"
extern "C" void rows(int m, int M, long stride, int K, unsigned elem_bytes, unsigned long* out) {
  const BufferRows r = buffer_rows(m, M, (size_t)stride, K, elem_bytes);
  out[0] = r.first; out[1] = r.bytes;
}
"""


@pytest.fixture(scope="module")
def buffer_rows(tmp_path_factory):
    folder = tmp_path_factory.mktemp("buffer")
    (folder / "host.cpp").write_text(HOST)
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-I", B.CSRC, str(folder / "host.cpp"), "-o", str(folder / "host.so")],
                   check=True, timeout=120)
    lib = ctypes.CDLL(str(folder / "host.so"))
    lib.rows.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_int, ctypes.c_uint, ctypes.c_void_p]

    def of(m, M, stride, K, size):
        out = (ctypes.c_ulong * 2)()
        lib.rows(m, M, stride, K, size, out)
        return out[0], out[1]
    return of


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_chains_of_32_bit_products_have_no_scalar_place(device_code, dtype):
    """Their lanes read on behind K, into the next row: of the last row only the range check stops them."""
    loads = re.findall(r"^\s*buffer_load_\S+ .*\], (\S+) offen", device_code("gemm.hip", dtype), re.M)
    assert len(loads) > 100 and set(loads) == {"0"}, set(loads)


@pytest.mark.parametrize("size", [4, 2])
@pytest.mark.parametrize("M, K, gap", [(1, 4, 0), (5, 36, 8), (17, 64, 0), (64, 292, 4), (130, 2052, 0), (3, 256, 0)])
def test_chains_read_their_rows_and_nothing_behind_the_last(buffer_rows, M, K, gap, size):
    stride, load = K + gap, 4 * size
    end = ((M - 1) * stride + K) * size
    for rows_a_block in (16, 64):
        for m0 in range(0, M, rows_a_block):
            first, total = buffer_rows(m0, M, stride, K, size)
            row = np.minimum(np.arange(rows_a_block), M - 1 - m0)[:, None]
            in_chain = np.arange(0, 32, 4)[None, :]
            for chain in range(-(-K // 32) + 16):               # a round's chains behind the last one too
                k = 32 * chain
                left = total - k * size if k < K else 0
                place = (row * stride + in_chain) * size
                reads = place < left
                assert left >= 0 and (place + load <= left)[reads].all()
                assert ((first + k) * size + place + load <= end)[reads].all()
                assert reads[np.broadcast_to(32 * chain + in_chain < K, reads.shape)].all()


@pytest.mark.parametrize("M, K, gap", [(1, 64, 0), (64, 128, 8), (65, 192, 0), (129, 320, 8), (200, 64, 64), (256, 128, 0), (333, 2048, 0)])
def test_tiles_read_rows_that_there_are(buffer_rows, M, K, gap):
    """Rows past M, whole groups of them too: a lane reads within the operand with its scalar place, or is stopped without it."""
    stride, block_rows, group = K + gap, 256, 64                 # rows of X a block, rows that the waves load at a time
    end = ((M - 1) * stride + K) * 2
    row, slot = np.arange(group)[:, None], np.arange(8)[None, :]
    place = (row * stride + slot * 8) * 2
    for m in range(0, -(-M // block_rows) * block_rows, group):
        first, total = buffer_rows(m, M, stride, K, 2)
        reads = place < total
        for k in range(0, K, 64):
            assert (place + 2 * k + 16 <= total)[reads].all() and (first * 2 + place + 2 * k + 16 <= end)[reads].all()
        assert (reads[np.broadcast_to(m + row < M, reads.shape)]).all()
        assert total > 0, "nothing is known of a scalar place in a buffer of no bytes"
