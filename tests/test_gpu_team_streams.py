"""Textures on callers' streams around the block counts where the direct
kernels change the number of groups that share a block there, several calls in
flight at once, against the oracle."""
import ctypes

import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["tx_compress_device", "tx_compress_device_noalloc"])
@pytest.mark.parametrize("fmt", [tx.Format.Bc1, tx.Format.Bc3], ids=lambda f: f.name)
def test_team_sizes_on_streams(gpu, oracle, fmt, entry):
    hip = ctypes.CDLL("libamdhip64.so")
    p = tx.Params(tx.Algorithm.IterativeClusterFit)
    op = oracle.params(2, p.weights, False)
    cp = p._c()
    calls = []
    for n in (7167, 7168, 7169, 10241):
        img = texgen.with_alpha_field(texgen.rgb_texture(4 * n, 4, n), n)
        want = oracle.compress(int(fmt), img, 4 * n, 4, op, threads=8)
        stream = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
        calls.append((n, stream, tx.DeviceBuffer.from_array(img),
                      tx.DeviceBuffer.from_array(np.full(want.size, 0x5A, np.uint8)), want))
    for n, stream, src, out, want in calls:
        assert getattr(gpu, entry)(int(fmt), src.ptr, 4 * n, 4, ctypes.byref(cp), out.ptr, want.size, stream) == 0
    for n, stream, src, out, want in calls:
        assert hip.hipStreamSynchronize(stream) == 0
        np.testing.assert_array_equal(out.download(), want, err_msg="%d blocks" % n)
        assert hip.hipStreamDestroy(stream) == 0
