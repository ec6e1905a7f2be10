"""A texture with more blocks than there is device memory for the pipeline's
records is encoded by the direct kernels, and the next one that has room takes
the pipeline again."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu


def test_more_blocks_than_records_fit(gpu, oracle):
    # an output of 2^30 + 1 blocks (8 GiB), nearly all of them past a 64 x 4
    # image and so fully masked; their records would take 2^31 * 232 bytes
    fmt, p = tx.Format.Bc1, tx.Params()
    nblocks = (1 << 30) + 1
    img = texgen.with_alpha_field(texgen.rgb_texture(64, 4, 5), 5)
    op = oracle.params(int(p.algorithm), p.weights, False)
    first = oracle.compress(int(fmt), img, 64, 4, op)
    empty = oracle.compress_blocks(int(fmt), np.zeros((1, 64), np.uint8), np.zeros(1, np.uint32), op)[0]
    src, out = tx.DeviceBuffer.from_array(img), tx.DeviceBuffer(8 * nblocks)
    fmt.compress_device(src.ptr, 64, 4, p, out.ptr, 8 * nblocks)
    np.testing.assert_array_equal(out.download(first.size), first)
    piece = np.empty(64 << 20, np.uint8)
    want = np.tile(empty, piece.size // 8)
    starts = list(range(first.size, 8 * nblocks - piece.size, 1 << 30)) + [8 * nblocks - piece.size]
    for at in starts:
        assert gpu.tx_util_download(piece.ctypes.data, out.ptr + at, piece.size) == 0
        np.testing.assert_array_equal(piece, want, err_msg="bytes from %d" % at)
    out.free()

    w, h = 640, 516
    img = texgen.with_alpha_field(texgen.rgb_texture(w, h, 6), 6)
    n = fmt.compressed_size(w, h)
    src, out = tx.DeviceBuffer.from_array(img), tx.DeviceBuffer(n)
    assert tx.time_phases(fmt, src.ptr, w, h, p, out.ptr, n, 1) is not None
    np.testing.assert_array_equal(out.download(), oracle.compress(int(fmt), img, w, h, op, threads=8))
