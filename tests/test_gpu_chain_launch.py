"""compress_mips_device encodes the levels of a chain in one launch: every
level must equal the same level compressed alone, for every format and
algorithm, on the direct kernels and through the pipeline, for chains of one
level, of sides of 1, of ragged levels and cut short."""
import numpy as np
import pytest

import texpresso_amd as tx
from texpresso_amd import texgen

pytestmark = pytest.mark.gpu

CASES = [(8, 8, None), (1, 9, None), (257, 3, None), (130, 61, 3), (500, 375, None), (33, 70, 1)]


def chain_bytes(fmt, img, levels, p, stream=None):
    h, w = img.shape[:2]
    src = tx.DeviceBuffer.from_array(img)
    chain = tx.DeviceBuffer(max(4, tx.mip_chain_rgba_bytes(w, h, levels)))
    n = fmt.mip_chain_size(w, h, levels)
    out = tx.DeviceBuffer.from_array(np.full(n + 64, 0x5A, np.uint8))
    fmt.compress_mips_device(src.ptr, w, h, p, levels, chain.ptr, chain.nbytes, out.ptr, n)
    got = out.download()
    assert (got[n:] == 0x5A).all()
    return got[:n]


@pytest.mark.parametrize("fmt", list(tx.Format), ids=lambda f: f.name)
@pytest.mark.parametrize("alg", list(tx.Algorithm), ids=lambda a: a.name)
@pytest.mark.parametrize("threshold", [0, 2**64 - 1], ids=["pipeline", "direct"])
def test_chain_equals_its_levels(gpu, oracle, fmt, alg, threshold):
    p = tx.Params(alg, tx.COLOUR_WEIGHTS_PERCEPTUAL, fmt == tx.Format.Bc2)
    op = oracle.params(int(alg), p.weights, p.weigh_colour_by_alpha)
    old = tx.set_pipeline_threshold(threshold)
    try:
        for w, h, levels in CASES:
            img = texgen.with_alpha_field(texgen.rgb_texture(w, h, w * 7 + h), w)
            levels = levels or tx.mip_levels(w, h)
            got = chain_bytes(fmt, img, levels, p)
            want = [oracle.compress(int(fmt), lv, lv.shape[1], lv.shape[0], op, threads=8)
                    for lv in texgen.mip_chain(img)[:levels]]
            np.testing.assert_array_equal(got, np.concatenate(want), err_msg=str((w, h, levels)))
    finally:
        tx.set_pipeline_threshold(old)
