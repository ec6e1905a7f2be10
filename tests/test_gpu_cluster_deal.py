"""ClusterFit record lists on both sides of the length from which the cluster
kernel takes its steps from the shared cursor (64 records a workgroup; 1024
workgroups on a card of 256 CUs), and around one step and one round of steps:
every block equals the direct kernels' block."""
import numpy as np
import pytest

import texpresso_amd as tx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc3])
@pytest.mark.parametrize("blocks", [1, 4, 5, 4096, 4097, 16384, 16385, 65535, 65536, 65537, 70001])
def test_list_lengths(fmt, blocks):
    # 64 colours: no flat block, so every block is one record
    rng = np.random.default_rng(blocks)
    img = (rng.integers(0, 4, (4, 4 * blocks, 4)) * 60).astype(np.uint8)
    img[..., 3] = 255
    params = tx.Params(tx.Algorithm.ClusterFit)
    src = tx.DeviceBuffer.from_array(img)
    n = fmt.compressed_size(4 * blocks, 4)
    out = tx.DeviceBuffer(n)
    got = []
    old = tx.set_pipeline_threshold(0)
    try:
        for threshold in (0, 2**64 - 1):  # pipeline, direct kernels
            tx.set_pipeline_threshold(threshold)
            out.upload(np.full(n, 0xA5, np.uint8))
            fmt.compress_device(src.ptr, 4 * blocks, 4, params, out.ptr, n)
            got.append(out.download())
    finally:
        tx.set_pipeline_threshold(old)
    np.testing.assert_array_equal(got[0], got[1])
