"""The decoder against the oracle at the widths where its tiling and its
stores change (one block to several waves across, widths that are no multiple
of 4), and from block data at every byte alignment."""
import numpy as np
import pytest

import texpresso_amd as tx

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (2, 9), (4, 4), (7, 70), (33, 18), (64, 3), (130, 37), (255, 5), (257, 21), (1023, 13)]


@pytest.mark.parametrize("fmt", list(tx.Format), ids=lambda f: f.name)
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_decode_sizes_and_alignments(gpu, oracle, fmt, offset):
    rng = np.random.default_rng(int(fmt) * 7 + offset)
    for w, h in SIZES:
        n = fmt.compressed_size(w, h)
        data = rng.integers(0, 256, n).astype(np.uint8)
        data[: n // 2 : 3] = 0  # equal endpoints and index runs among the random ones
        src = tx.DeviceBuffer(n + offset)
        src.upload(np.concatenate([np.full(offset, 0xA5, np.uint8), data]))
        dst = tx.DeviceBuffer.from_array(np.full(4 * w * h + 16, 0x5A, np.uint8))
        fmt.decompress_device(src.ptr + offset, w, h, dst.ptr)
        got = dst.download()
        np.testing.assert_array_equal(got[: 4 * w * h], oracle.decompress(int(fmt), data, w, h), err_msg=str((w, h)))
        assert (got[4 * w * h :] == 0x5A).all(), "bytes past the image were written"
