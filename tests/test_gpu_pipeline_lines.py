"""The block counts from which a texture on the library's own stream goes
through the binned pipeline, by format, algorithm and weighting, and its bytes
on both sides of each line, against the oracle."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

# (algorithm, weighed by alpha): first block count of the pipeline, BC1 and BC2/BC3
LINES = {(1, False): (18432, 18432), (1, True): (28672, 40960), (2, False): (98304, 32768), (2, True): (98304, 32768)}


@pytest.mark.parametrize("alg,weighed", LINES, ids=lambda v: str(v))
@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc3], ids=lambda f: f.name)
def test_pipeline_lines(gpu, oracle, fmt, alg, weighed):
    line = LINES[alg, weighed][0 if fmt == tx.Format.Bc1 else 1]
    p = tx.Params(tx.Algorithm(alg), tx.COLOUR_WEIGHTS_PERCEPTUAL, weighed)
    op = oracle.params(alg, p.weights, weighed)
    base = texgen.with_alpha_field(texgen.rgb_texture(1024, 16, line), line)
    base[:, 256:768] = base[:4, 256:260].repeat(4, 0).repeat(128, 1)  # half of it flat in rows
    for w, h, piped in ((1024, line // 64 - 4, False), (1024, line // 64, True)):
        img = np.ascontiguousarray(np.tile(base, (h // 16 + 1, 1, 1))[:h])
        n = fmt.compressed_size(w, h)
        assert n // fmt.block_size() == line - (0 if piped else 256)
        src, out = tx.DeviceBuffer.from_array(img), tx.DeviceBuffer(n)
        assert (tx.time_phases(fmt, src.ptr, w, h, p, out.ptr, n, 1) is not None) == piped
        want = oracle.compress(int(fmt), img[:16], w, 16, op, threads=8)
        got = out.download().reshape(-1, want.size // 4)  # rows of blocks: the image repeats every four
        for row in range(len(got)):
            np.testing.assert_array_equal(got[row], want.reshape(4, -1)[row % 4], err_msg="row %d" % row)
