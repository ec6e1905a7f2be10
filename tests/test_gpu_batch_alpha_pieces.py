"""Batches of BC4/BC5 textures with as many chunks as lie around the counts
where the chunks are cut coarser, and where they are first drawn from the
counter, against the oracle, on repeated runs."""
import numpy as np
import pytest

import texpresso_amd as tx
from tests.blockgen import make_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [tx.Format.Bc4, tx.Format.Bc5], ids=lambda f: f.name)
@pytest.mark.parametrize("count", [1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193])
def test_alpha_chunk_counts(gpu, oracle, fmt, count):
    blocks, _ = make_blocks(4096, per_class=64)
    sizes = 1 + np.arange(count) % 3  # blocks of each texture, one row high
    sizes[0], sizes[1] = 512, 130  # a whole chunk and a part of one
    ends = np.cumsum(sizes)
    pick = np.random.default_rng(count).integers(0, len(blocks), ends[-1])
    src_blocks = blocks[pick].reshape(-1, 4, 4, 4)
    rows = [src_blocks[e - n : e].transpose(1, 0, 2, 3).reshape(-1) for e, n in zip(ends, sizes)]
    src = tx.DeviceBuffer.from_array(np.concatenate(rows))
    want = oracle.compress_blocks(int(fmt), blocks[pick], np.full(len(pick), 0xFFFF, np.uint32), oracle.params())
    out = tx.DeviceBuffer(want.size)
    bs = fmt.block_size()
    items = [(fmt, tx.Params(), src.ptr + 64 * int(e - n), out.ptr + bs * int(e - n), 4 * int(n), 4)
             for e, n in zip(ends, sizes)]
    for graph in (True, False):
        batch = tx.Batch(items, tx.Tuning(use_graph=graph))
        for run in range(3):
            out.upload(np.full(want.size, run, np.uint8))
            batch.run()
            np.testing.assert_array_equal(out.download().reshape(want.shape), want, err_msg="run %d" % run)
        batch.close()
