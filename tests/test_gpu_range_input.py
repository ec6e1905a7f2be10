"""RangeFit textures around the block counts where the direct kernel changes
from a 16-lane group per block to a block per lane, from host memory (which the
kernels read over the bus) and from device memory, against the oracle."""
import numpy as np
import pytest

import texpresso_amd as tx
from tests.test_gpu_range_lines import SHAPES
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

HOST = [(n, short, h) for n in (1, 256, 512, 513, 1280, 1281, 4096) for short in (0, 1) for h in (4, 7)]


def _check(oracle, fmt, weighed, shapes, encode):
    p = tx.Params(tx.Algorithm.RangeFit, tx.COLOUR_WEIGHTS_PERCEPTUAL, weighed)
    op = oracle.params(0, p.weights, weighed)
    for n, short, h in shapes:
        w = 4 * n - short
        img = texgen.with_alpha_field(texgen.rgb_texture(w, h, n), n)
        img[:, ::7] = img[:, :1]  # blocks of few colours among them
        want = oracle.compress(int(fmt), img, w, h, op, threads=8).reshape(-1)
        np.testing.assert_array_equal(encode(img, w, h, p, want.size), want, err_msg="%d x %d" % (w, h))


@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc2, tx.Format.Bc3], ids=lambda f: f.name)
@pytest.mark.parametrize("weighed", [False, True], ids=["plain", "weighed"])
def test_from_host(gpu, oracle, fmt, weighed):
    def encode(img, w, h, p, size):
        got = np.zeros(size, np.uint8)
        fmt.compress(img, w, h, p, got)
        return got

    _check(oracle, fmt, weighed, HOST, encode)


@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc2, tx.Format.Bc3], ids=lambda f: f.name)
@pytest.mark.parametrize("kind", SHAPES)
def test_from_device(gpu, oracle, fmt, kind):
    def encode(img, w, h, p, size):
        src, out = tx.DeviceBuffer.from_array(img), tx.DeviceBuffer(size)
        fmt.compress_device(src.ptr, w, h, p, out.ptr, size)
        return out.download()

    _check(oracle, fmt, kind == "weighed", SHAPES[kind], encode)
