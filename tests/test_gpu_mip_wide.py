"""Mip levels of an image so wide that a row of its tiles is past a launch's
limit of work-items and takes several launches."""
import numpy as np
import pytest

import texpresso_amd as tx

pytestmark = pytest.mark.gpu


def test_widest_levels(gpu):
    """2^30 + 6 texels in one row (4 GiB) and its first three levels.  The row
    repeats a pattern whose length has no more factors of 2 than the levels
    need, so that a misplaced tile shows."""
    w, period, levels = (1 << 30) + 6, 15000008, 4
    level = np.random.default_rng(1).integers(0, 256, (period, 4), dtype=np.uint8)
    n = tx.mip_chain_rgba_bytes(w, 1, levels)
    src, dst = tx.DeviceBuffer(4 * w), tx.DeviceBuffer(n)
    for at in range(0, w, period):
        assert gpu.tx_util_upload(src.ptr + 4 * at, level.ctypes.data, 4 * min(period, w - at)) == 0
    tx.generate_mips_device(src.ptr, w, 1, levels, dst.ptr, n)
    got, ptr = np.empty((period, 4), np.uint8), dst.ptr
    for k in range(1, levels):
        pair = level.reshape(-1, 2, 4).astype(np.uint16)
        level = ((2 * (pair[:, 0] + pair[:, 1]) + 2) >> 2).astype(np.uint8)
        for at in range(0, w >> k, len(level)):
            count = min(len(level), (w >> k) - at)
            assert gpu.tx_util_download(got.ctypes.data, ptr + 4 * at, 4 * count) == 0
            np.testing.assert_array_equal(got[:count], level[:count], err_msg="level %d from %d" % (k, at))
        ptr += 4 * (w >> k)
    assert ptr == dst.ptr + n
    src.free()
    dst.free()
