"""The split search's reciprocal, as the device evaluates it, against numpy's
correctly rounded binary32 division, bit for bit: every significand at every
exponent that a split's determinant can have, and at the ends of the range for
which the reciprocal is exact, both signs, and the special values.

A determinant is alpha2_sum * beta2_sum - alphabeta_sum^2 of point weights in
[1/16, 4] (sqrt of a pixel count, or of a sum of (alpha + 1) / 256): a product
of two sums below 64, each 0 or at least 1/144, so 0 or, as the difference of
two binary32 products of at least 2^-20, at least 2^-44, and below 2^12."""
import numpy as np
import pytest

import texpresso_amd as tx

pytestmark = pytest.mark.gpu

SIGNIFICANDS = np.arange(1 << 23, dtype=np.uint32)


def check(exponent, sign):
    bits = SIGNIFICANDS | np.uint32((exponent + 127) << 23) | np.uint32(0x80000000 if sign < 0 else 0)
    x = bits.view(np.float32)
    want = np.float32(1) / x
    bad = np.flatnonzero(tx.reciprocal(x).view(np.uint32) != want.view(np.uint32))
    assert bad.size == 0, "2^%d: %d differ, first at %r" % (exponent, bad.size, x[bad[0]])


@pytest.mark.parametrize("sign", [1, -1])
def test_every_determinant(gpu, sign):
    for exponent in range(-45, 14):
        check(exponent, sign)


@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("exponent", [-126, -125, -64, 64, 124, 125])
def test_ends_of_the_range(gpu, exponent, sign):
    check(exponent, sign)


def test_special_values(gpu):
    x = np.array([0.0, -0.0, np.inf, -np.inf], np.float32)
    with np.errstate(divide="ignore"):
        want = np.float32(1) / x
    np.testing.assert_array_equal(tx.reciprocal(x).view(np.uint32), want.view(np.uint32))
    assert np.isnan(tx.reciprocal(np.array([np.nan], np.float32))).all()
