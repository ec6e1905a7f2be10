"""A mip chain whose first level has more than 2^20 blocks: that level goes on
its own and the others together, and each is what it is alone."""
import ctypes

import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

W, H = 4103, 4098  # 1026 x 1025 blocks


@pytest.mark.parametrize("stream", ["library", "caller"])
@pytest.mark.parametrize("fmt,alg", [(tx.Format.Bc1, 0), (tx.Format.Bc1, 1), (tx.Format.Bc3, 2), (tx.Format.Bc4, 0)],
                         ids=["bc1-range", "bc1-cluster", "bc3-iterative", "bc4"])
def test_large_level(gpu, oracle, fmt, alg, stream):
    assert tx.num_blocks(W) * tx.num_blocks(H) > 1 << 20
    base = texgen.with_alpha_field(texgen.rgb_texture(513, 514, 11), 11)
    img = np.ascontiguousarray(np.tile(base, (8, 8, 1))[:H, :W])
    p, levels = tx.Params(tx.Algorithm(alg)), tx.mip_levels(W, H)
    mips = texgen.mip_chain(img)
    src = tx.DeviceBuffer.from_array(img)
    chain = tx.DeviceBuffer(tx.mip_chain_rgba_bytes(W, H, levels))
    out = tx.DeviceBuffer.from_array(np.full(fmt.mip_chain_size(W, H, levels) + 64, 0x5A, np.uint8))
    handle = ctypes.c_void_p()
    hip = ctypes.CDLL("libamdhip64.so")
    if stream == "caller":
        assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0
    fmt.compress_mips_device(src.ptr, W, H, p, levels, chain.ptr, chain.nbytes, out.ptr, out.nbytes - 64, handle)
    assert hip.hipDeviceSynchronize() == 0
    got = out.download()
    np.testing.assert_array_equal(chain.download(), np.concatenate([m.reshape(-1) for m in mips[1:]]))
    op = oracle.params(alg, p.weights, False)
    at, from_chain = 0, 0
    for k, m in enumerate(mips):
        h, w = m.shape[:2]
        n = fmt.compressed_size(w, h)
        alone = tx.DeviceBuffer(n)
        level = src.ptr if k == 0 else chain.ptr + from_chain
        fmt.compress_device(level, w, h, p, alone.ptr, n)
        assert hip.hipDeviceSynchronize() == 0
        np.testing.assert_array_equal(got[at : at + n], alone.download(), err_msg="level %d alone" % k)
        # the oracle: whole small levels, and the first and last rows of blocks of the others
        for rows in [slice(0, h)] if k >= 4 else [slice(0, 8), slice((h - 1) // 4 * 4, h)]:
            part = np.ascontiguousarray(m[rows])
            want = oracle.compress(int(fmt), part, w, part.shape[0], op, threads=8)
            first = at + fmt.compressed_size(w, rows.start)
            np.testing.assert_array_equal(got[first : first + want.size], want, err_msg="level %d" % k)
        at += n
        from_chain += 0 if k == 0 else 4 * w * h
    assert (got[at:] == 0x5A).all()
    if stream == "caller":
        assert hip.hipStreamDestroy(handle) == 0
