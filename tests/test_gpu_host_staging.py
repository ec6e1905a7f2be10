"""Host-buffer calls around the sizes where their input and output change
between the pinned memory, a copy from it and a copy from the caller's memory,
one call after another with other data, against the oracle."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

# 4 bytes a pixel: around 32 KiB and 1 MiB of input
SIZES = [(1, 1), (91, 90), (128, 64), (129, 64), (512, 511), (512, 512), (516, 512), (1024, 513)]


@pytest.mark.parametrize("fmt,alg", [(tx.Format.Bc1, 0), (tx.Format.Bc3, 1), (tx.Format.Bc5, 0)],
                         ids=["bc1_range", "bc3_cluster", "bc5"])
def test_staged_calls(gpu, oracle, fmt, alg):
    p = tx.Params(tx.Algorithm(alg))
    op = oracle.params(alg, p.weights, False)
    for w, h in SIZES + SIZES[::-1]:
        img = texgen.with_alpha_field(texgen.rgb_texture(w, h, w + h), h)
        want = oracle.compress(int(fmt), img, w, h, op, threads=8)
        got = np.zeros_like(want)
        fmt.compress(img, w, h, p, got)
        np.testing.assert_array_equal(got, want, err_msg="encode %dx%d" % (w, h))
        pixels = np.zeros(4 * w * h, np.uint8)
        fmt.decompress(got, w, h, pixels)
        np.testing.assert_array_equal(pixels, oracle.decompress(int(fmt), want, w, h), err_msg="decode %dx%d" % (w, h))
        levels = min(3, tx.mip_levels(w, h))
        chain = [oracle.compress(int(fmt), lv, lv.shape[1], lv.shape[0], op, threads=8)
                 for lv in texgen.mip_chain(img)[:levels]]
        np.testing.assert_array_equal(fmt.compress_mips(img, w, h, p, levels), np.concatenate(chain))


@pytest.mark.parametrize("n", [481, 482, 483, 15420, 15421])  # 68 bytes in each: around 32 KiB and 1 MiB
def test_staged_block_lists(gpu, oracle, n):
    rng = np.random.default_rng(n)
    blocks = rng.integers(0, 256, (n, 64)).astype(np.uint8)
    masks = rng.integers(0, 1 << 16, n).astype(np.uint32)
    p = tx.Params(tx.Algorithm.RangeFit)
    want = oracle.compress_blocks(0, blocks, masks, oracle.params(0, p.weights, False))
    np.testing.assert_array_equal(tx.compress_blocks(tx.Format.Bc1, blocks, masks, p), want)
