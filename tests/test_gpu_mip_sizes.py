"""Mip levels at the sizes where the tiled kernel can go wrong: around its
64-texel tiles and their halves, sides of 1, odd sides, chains longer than one
launch and chains cut short, with the bytes past the chain left alone."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

SIZES = [(2, 1), (1, 2), (3, 3), (1, 300), (300, 1), (2, 129), (5, 64), (63, 65), (64, 64), (65, 127), (128, 192),
         (130, 31), (257, 255), (1000, 7), (511, 1025)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "%dx%d" % s)
def test_mip_sizes(gpu, size):
    w, h = size
    img = np.random.default_rng(w * 4099 + h).integers(0, 256, (h, w, 4)).astype(np.uint8)
    want = texgen.mip_chain(img)[1:]
    src = tx.DeviceBuffer.from_array(img)
    for levels in sorted({2, 3, 4, len(want), len(want) + 1}):
        if not 2 <= levels <= len(want) + 1:
            continue
        n = tx.mip_chain_rgba_bytes(w, h, levels)
        dst = tx.DeviceBuffer.from_array(np.full(n + 16, 0x5A, np.uint8))
        tx.generate_mips_device(src.ptr, w, h, levels, dst.ptr, n)
        got = dst.download()
        at = 0
        for k, level in enumerate(want[: levels - 1]):
            np.testing.assert_array_equal(got[at : at + level.size].reshape(level.shape), level,
                                          err_msg="level %d of %d" % (k + 1, levels))
            at += level.size
        assert at == n and (got[n:] == 0x5A).all()
