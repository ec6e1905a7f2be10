"""The split search for every colour count: blocks of exactly n distinct
colours (n = 2..16), with equal steps (exact ties between splits), random and
clustered colours, every pixel of one colour or the spare pixels repeated,
against the oracle, through the direct kernel and the binned pipeline."""
import numpy as np
import pytest

import texpresso_amd as tx

pytestmark = pytest.mark.gpu


def blocks_of(n, seed, per_kind=24):
    rng = np.random.default_rng(seed * 31 + n)
    out = []
    for kind in ("steps", "random", "clusters") * per_kind:
        if kind == "steps":  # equal steps along a line
            d = rng.integers(1, 4, 3) * rng.choice([-1, 1], 3)
            cols = rng.integers(60, 190, 3) + np.arange(n)[:, None] * d
        elif kind == "random":
            cols = rng.permutation(256)[:n, None] * np.array([1, 0, 0]) + rng.integers(0, 256, (n, 3)) * [0, 1, 1]
        else:  # two tight clusters
            far = rng.integers(0, 2, n)[:, None] * rng.integers(60, 120, 3)
            cols = rng.integers(20, 120, 3) + far + np.stack([np.arange(n), np.zeros(n), rng.permutation(n)], 1)
        pick = np.concatenate([np.arange(n), rng.integers(0, n, 16 - n)])
        px = np.zeros((16, 4), np.uint8)
        px[:, :3] = np.clip(cols, 0, 255).astype(np.uint8)[rng.permutation(pick)]
        px[:, 3] = 255 if rng.random() < 0.5 else rng.choice([40, 130, 200, 255], 16)
        out.append(px)
    return np.stack(out)


@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc3], ids=lambda f: f.name)
@pytest.mark.parametrize("alg", [tx.Algorithm.ClusterFit, tx.Algorithm.IterativeClusterFit], ids=lambda a: a.name)
@pytest.mark.parametrize("by_alpha", [False, True], ids=["plain", "by_alpha"])
def test_every_colour_count(gpu, oracle, fmt, alg, by_alpha):
    p = tx.Params(alg, tx.COLOUR_WEIGHTS_PERCEPTUAL, by_alpha)
    op = oracle.params(int(alg), p.weights, by_alpha)
    blocks = np.concatenate([blocks_of(n, 5) for n in range(2, 17)])
    masks = np.full(len(blocks), 0xFFFF, np.uint32)
    want = oracle.compress_blocks(int(fmt), blocks, masks, op)
    np.testing.assert_array_equal(tx.compress_blocks(fmt, blocks, masks, p), want)
    # the same blocks side by side as one texture row, through the pipeline
    img = np.ascontiguousarray(blocks.reshape(-1, 4, 4, 4).transpose(1, 0, 2, 3)).reshape(4, -1, 4)
    got = np.zeros(want.size, np.uint8)
    old = tx.set_pipeline_threshold(0)
    try:
        fmt.compress(img, img.shape[1], 4, p, got)
    finally:
        tx.set_pipeline_threshold(old)
    np.testing.assert_array_equal(got.reshape(want.shape), want)
