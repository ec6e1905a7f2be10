"""Batches and servers with chunk sizes far above their textures, up to the
largest that a tuning may name (2^32 - 4: never split): every texture's bytes
are the oracle's, with fewer chunks than waves and with more, on the lockstep
kernels and on the pipeline."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

CHUNKS = [1 << 20, (1 << 31) - 4, (1 << 31) + 4, 0xFFFFFFC0, 0xFFFFFFC4, 0xFFFFFFFC]
KINDS = [(tx.Format.Bc1, 1), (tx.Format.Bc3, 2), (tx.Format.Bc2, 0), (tx.Format.Bc4, 0)]


@pytest.fixture(scope="module")
def textures(gpu, oracle):
    rows = []
    for i, (w, h) in enumerate([(4, 4), (60, 12), (257, 9), (129, 64)]):
        img = texgen.with_alpha_field(texgen.rgb_texture(w, h, i), i)
        src = tx.DeviceBuffer.from_array(img)
        for fmt, alg in KINDS:
            p = tx.Params(tx.Algorithm(alg))
            rows.append((fmt, p, img, src, oracle.compress(int(fmt), img, w, h, oracle.params(alg, p.weights, False))))
    return rows


@pytest.mark.parametrize("pipeline", [False, True], ids=["lockstep", "pipeline"])
@pytest.mark.parametrize("chunk", CHUNKS)
@pytest.mark.parametrize("copies,waves,lanes,graph", [(1, 1, 1, True), (30, 4, 16, False)], ids=["few", "many"])
def test_batch_chunk_sizes(textures, pipeline, chunk, copies, waves, lanes, graph):
    # many: 360 colour chunks on at most 256 workgroups of one wave
    groups = 12 if copies == 1 else 1
    items, outs = [], []
    for fmt, p, img, src, ref in textures * copies:
        out = tx.DeviceBuffer.from_array(np.full(ref.size, 0x5A, np.uint8))
        items.append((fmt, p, src.ptr, out.ptr, img.shape[1], img.shape[0]))
        outs.append((out, ref))
    for w in {1, waves}:
        batch = tx.Batch(items, tx.Tuning(chunk, w, groups, graph, pipeline, lanes))
        # one chunk each, but alpha-only textures have 512-block chunks with one lane a block
        alpha = [tx.num_blocks(i[4]) * tx.num_blocks(i[5]) for i in items if i[0] == tx.Format.Bc4 and lanes == 1]
        assert batch.info()["chunks"] == len(items) - len(alpha) + sum((n + 511) // 512 for n in alpha)
        for run in range(2):
            batch.run()
            for out, ref in outs:
                np.testing.assert_array_equal(out.download(), ref, err_msg="waves %d run %d" % (w, run))
                out.upload(np.full(ref.size, run, np.uint8))
        batch.close()


@pytest.mark.parametrize("chunk", [4, 128, 0xFFFFFFFC])
@pytest.mark.parametrize("threshold", [0, 2**64 - 1], ids=["pipeline", "lockstep"])
def test_server_chunk_sizes(textures, chunk, threshold):
    old = tx.set_pipeline_threshold(threshold)
    try:
        server = tx.Server(hbm_budget=64 << 20, tuning=tx.Tuning(chunk_blocks=chunk, pipeline=True))
        ids = [server.submit(fmt, img, img.shape[1], img.shape[0], p) for fmt, p, img, _, _ in textures * 3]
        for jid, (_, _, _, _, ref) in zip(ids, textures * 3):
            assert server.wait(jid).status == 3
            np.testing.assert_array_equal(server.fetch(jid, ref.size), ref)
            server.release(jid)
        server.close()
    finally:
        tx.set_pipeline_threshold(old)
