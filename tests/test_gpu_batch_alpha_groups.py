"""Batches of colour and BC4/BC5 textures whose alpha-only chunks take 16 lanes
a block, beside each colour path, against the oracle, on repeated runs: the
searches of the binned pipeline start after the alpha kernel has ended."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

SIZES = [(64, 64), (131, 77), (5, 3), (256, 40), (3, 90), (160, 200)]


@pytest.mark.parametrize("graph", [True, False], ids=["graph", "plain"])
@pytest.mark.parametrize("pipeline", [True, False], ids=["pipeline", "lockstep"])
@pytest.mark.parametrize("alg", list(tx.Algorithm), ids=lambda a: a.name)
def test_alpha_groups_beside_colour(gpu, oracle, alg, pipeline, graph):
    items, outs, want, keep = [], [], [], []
    for k, (w, h) in enumerate(SIZES):
        img = texgen.with_alpha_field(texgen.rgb_texture(w, h, 50 + k), 50 + k)
        src = tx.DeviceBuffer.from_array(img)
        keep.append(src)
        for fmt in tx.Format:
            out = tx.DeviceBuffer(fmt.compressed_size(w, h))
            p = tx.Params(alg)
            items.append((fmt, p, src.ptr, out.ptr, w, h))
            outs.append(out)
            want.append(oracle.compress(int(fmt), img, w, h, oracle.params(int(alg), p.weights, False)).reshape(-1))
    batch = tx.Batch(items, tx.Tuning(chunk_blocks=32, use_graph=graph, pipeline=pipeline, lanes_per_block=16))
    for run in range(3):
        for out in outs:
            out.upload(np.full(out.nbytes, run, np.uint8))
        batch.run()
        for item, out, w in zip(items, outs, want):
            np.testing.assert_array_equal(out.download(), w, err_msg="run %d %s %dx%d" % (run, item[0].name, item[4],
                                                                                          item[5]))
    batch.close()
