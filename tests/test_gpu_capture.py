"""Encodes captured into a graph on a caller's stream, above and below the
block counts where the same calls use the binned pipeline outside a capture:
every replay, on new pixels, gives the oracle's bytes."""
import ctypes

import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,alg,size", [(tx.Format.Bc1, 1, (640, 300)), (tx.Format.Bc3, 1, (1000, 900)),
                                          (tx.Format.Bc4, 0, (129, 77))], ids=["small", "large", "bc4"])
def test_captured_encode_and_chain(gpu, oracle, fmt, alg, size):
    w, h = size
    p = tx.Params(tx.Algorithm(alg))
    op = oracle.params(alg, p.weights, False)
    levels, n = tx.mip_levels(w, h), fmt.compressed_size(w, h)
    src, out = tx.DeviceBuffer(4 * w * h), tx.DeviceBuffer(n)
    chain = tx.DeviceBuffer(tx.mip_chain_rgba_bytes(w, h, levels))
    mips = tx.DeviceBuffer(fmt.mip_chain_size(w, h, levels))
    # a call outside a capture first, so that what the library sets up once is there
    fmt.compress_device(src.ptr, w, h, p, out.ptr, n)
    hip = ctypes.CDLL("libamdhip64.so")
    stream, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local mode
    fmt.compress_device(src.ptr, w, h, p, out.ptr, n, stream)
    fmt.compress_mips_device(src.ptr, w, h, p, levels, chain.ptr, chain.nbytes, mips.ptr, mips.nbytes, stream)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for seed in range(3):
        img = texgen.with_alpha_field(texgen.rgb_texture(w, h, seed), seed)
        src.upload(img.reshape(-1))
        out.upload(np.full(n, seed, np.uint8))
        mips.upload(np.full(mips.nbytes, seed, np.uint8))
        assert hip.hipGraphLaunch(run, stream) == 0
        assert hip.hipStreamSynchronize(stream) == 0
        want = [oracle.compress(int(fmt), lv, lv.shape[1], lv.shape[0], op, threads=8) for lv in texgen.mip_chain(img)]
        np.testing.assert_array_equal(out.download(), want[0], err_msg="replay %d" % seed)
        np.testing.assert_array_equal(mips.download(), np.concatenate(want), err_msg="chain, replay %d" % seed)
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(stream) == 0
