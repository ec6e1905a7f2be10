"""Textures around the block counts where the direct kernels change the
number of 16-lane groups that share a block, including last waves that are
partly empty, against the oracle."""
import numpy as np
import pytest

import texpresso_amd as tx
from tests.blockgen import make_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc2], ids=lambda f: f.name)
@pytest.mark.parametrize("alg,nblocks", [(1, 1), (1, 3), (1, 2560), (1, 2561), (1, 6143), (1, 6145),
                                         (2, 1), (2, 3), (2, 10240), (2, 10241), (2, 10243)])
def test_team_sizes(gpu, oracle, fmt, alg, nblocks):
    blocks, masks = make_blocks(nblocks, per_class=64)
    pick = np.random.default_rng(nblocks).integers(0, len(blocks), nblocks)
    blocks, masks = blocks[pick], masks[pick]
    p = tx.Params(tx.Algorithm(alg), tx.COLOUR_WEIGHTS_PERCEPTUAL, bool(nblocks & 1))
    op = oracle.params(alg, p.weights, p.weigh_colour_by_alpha)
    want = oracle.compress_blocks(int(fmt), blocks, masks, op)
    np.testing.assert_array_equal(tx.compress_blocks(fmt, blocks, masks, p), want)
    # unmasked, as a texture one block row high
    want = oracle.compress_blocks(int(fmt), blocks, np.full(nblocks, 0xFFFF, np.uint32), op)
    img = np.ascontiguousarray(blocks.reshape(-1, 4, 4, 4).transpose(1, 0, 2, 3)).reshape(4, -1, 4)
    got = np.zeros(want.size, np.uint8)
    fmt.compress(img, 4 * nblocks, 4, p, got)
    np.testing.assert_array_equal(got.reshape(want.shape), want)
