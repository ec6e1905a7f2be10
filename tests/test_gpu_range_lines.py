"""RangeFit textures around the block counts where the direct kernel changes
from a 16-lane group per block to a block per lane, by format, weighting and
shape, against the oracle."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

# one row of blocks: (blocks, pixels short of the last block's width, height)
SHAPES = {
    "full": [(n, 0, 4) for n in (1, 2560, 2561, 5120, 5121)],
    "ragged": [(n, 1, 4) for n in (1, 2560, 2561, 10240, 10241)],
    "thin": [(n, 0, h) for n in (8192, 8193) for h in (1, 3)],
    "weighed": [(n, short, 4) for n in (1, 12288, 12289) for short in (0, 3)],
}


@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc2, tx.Format.Bc3], ids=lambda f: f.name)
@pytest.mark.parametrize("kind", SHAPES)
def test_range_lines(gpu, oracle, fmt, kind):
    p = tx.Params(tx.Algorithm.RangeFit, tx.COLOUR_WEIGHTS_PERCEPTUAL, kind == "weighed")
    op = oracle.params(0, p.weights, p.weigh_colour_by_alpha)
    for n, short, h in SHAPES[kind]:
        w = 4 * n - short
        img = texgen.with_alpha_field(texgen.rgb_texture(w, h, n), n)
        img[:, ::7] = img[:, :1]  # blocks of few colours among them
        got = np.zeros(fmt.compressed_size(w, h), np.uint8)
        fmt.compress(img.reshape(-1), w, h, p, got)
        want = oracle.compress(int(fmt), img, w, h, op, threads=8)
        np.testing.assert_array_equal(got, want, err_msg="%d x %d" % (w, h))
