"""Batches whose chunks are cut into pieces: BC4/BC5 textures around one step
(64 blocks) and one chunk (512 blocks), colour textures in chunks below, at and
above 64 blocks, few and many of them, against the oracle, on repeated runs."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

# one block row: widths of 1, 63, 64, 65, 511, 512, 513 and 1100 blocks
BLOCKS = [1, 63, 64, 65, 511, 512, 513, 1100]


@pytest.mark.parametrize("pipeline", [False, True])
@pytest.mark.parametrize("chunk", [4, 64, 68, 128, 256])
@pytest.mark.parametrize("copies", [1, 40])
def test_batch_pieces(gpu, oracle, pipeline, chunk, copies):
    items, want, keep = [], [], []
    for i, n in enumerate(BLOCKS):
        img = texgen.with_alpha_field(texgen.rgb_texture(4 * n, 4, n), n)
        src = tx.DeviceBuffer.from_array(img)
        for fmt, alg in ((tx.Format.Bc4, 0), (tx.Format.Bc5, 0), (tx.Format.Bc1, 1 + i % 2), (tx.Format.Bc3, 0)):
            p = tx.Params(tx.Algorithm(alg))
            ref = oracle.compress(int(fmt), img, 4 * n, 4, oracle.params(alg, p.weights, False))
            for _ in range(copies):
                out = tx.DeviceBuffer.from_array(np.full(ref.size, 0x5A, np.uint8))
                items.append((fmt, p, src.ptr, out.ptr, 4 * n, 4))
                want.append(ref)
                keep.append((src, out))
    batch = tx.Batch(items, tx.Tuning(chunk_blocks=chunk, pipeline=pipeline))
    for run in range(3):
        batch.run()
        for (_, out), ref in zip(keep, want):
            np.testing.assert_array_equal(out.download(ref.size), ref, err_msg="run %d" % run)
            out.upload(np.full(ref.size, run, np.uint8))
    batch.close()
