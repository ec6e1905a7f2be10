"""Mip levels at the sizes where a few levels go by a launch each instead of in
tiles: one level of widths that are no multiple of 4, and a number of
levels that grows with the width, of wide images below 16 rows; with the bytes past the levels left alone."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

SIZES = [(61, 130), (65, 130), (66, 3), (131, 65), (1023, 66), (1 << 18, 1), ((1 << 18) + 3, 2), ((1 << 18) - 1, 5),
         (1 << 18, 15), ((1 << 18) + 1, 16), (1 << 18, 17), (1 << 19, 1), ((3 << 18) - 1, 2), ((3 << 18) + 1, 15),
         (6 << 18, 3)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "%dx%d" % s)
def test_levels(gpu, size):
    w, h = size
    img = np.random.default_rng(w * 31 + h).integers(0, 256, (h, w, 4), dtype=np.uint8)
    want = texgen.mip_chain(img)[1:]
    src = tx.DeviceBuffer.from_array(img)
    for levels in (2, 3, 4, 5, 7):
        n = tx.mip_chain_rgba_bytes(w, h, levels)
        dst = tx.DeviceBuffer.from_array(np.full(n + 16, 0x5A, np.uint8))
        tx.generate_mips_device(src.ptr, w, h, levels, dst.ptr, n)
        got = dst.download()
        np.testing.assert_array_equal(got[:n], np.concatenate([v.reshape(-1) for v in want[: levels - 1]]),
                                      err_msg="%d levels" % levels)
        assert (got[n:] == 0x5A).all()
