"""Pooling (csrc/pool.h): windows of every block of taps on each path of channels, windows that the image ends in on the right and below, that begin
in the padding and that lie outside altogether, and products of the average's requantisation on both sides of 32 bits."""
import numpy as np
import pytest

import oracle
from gpu_helpers import assert_same, avgpool, maxpool, rand_u8, rng_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels", [16, 48, 20, 7])
@pytest.mark.parametrize("kernel", [(1, 1), (2, 2), (3, 3), (2, 3), (4, 3), (4, 4), (5, 2), (7, 7), (2, 1), (1, 2), (3, 1), (1, 3), (1, 4), (5, 1),
                                    (5, 3), (6, 6), (7, 1), (1, 8), (10, 11)], ids=str)
def test_windows(kernel, channels):
    r = rng_for(8500 + 10 * kernel[0] + kernel[1] + channels)
    x = rand_u8(r, (3, 11, 13, channels))
    for strides in ((1, 1), (2, 3)):
        Ho, Wo = (11 - kernel[1]) // strides[1] + 1, (13 - kernel[0]) // strides[0] + 1
        for extra in (0, 1):  # one more row and column: windows that the image ends in
            out_hw = (Ho + extra, Wo + extra) if extra and (Ho * strides[1] < 11 and Wo * strides[0] < 13) else (Ho, Wo)
            assert_same(maxpool(x, kernel, strides, out_hw)[0], oracle.maxpool(x, kernel, strides, out_hw=out_hw), "max")
            for bits in (32, 64):
                for rq, lam, sh, ad in [(0, 0, 0, 0), (1, 300, 7, 900)] + ([(1, 2 ** 33 + 7, 34, 2 ** 36), (1, -5, 1, 400)] if bits == 64 else []):
                    want = oracle.avgpool(x, kernel, strides, (0, 0, 0, 0), out_hw, lam, sh, ad, rq, bits)
                    got = avgpool(x, kernel, strides, out_hw, (0, 0, 0, 0), lam, sh, ad, rq, bits)
                    assert_same(got, want, "average %s" % ((bits, rq, lam),))


@pytest.mark.parametrize("channels", [16, 48, 20, 7])
@pytest.mark.parametrize("kernel", [(2, 2), (1, 2), (2, 1), (3, 3), (2, 3), (4, 1), (1, 4), (5, 3), (4, 4)], ids=str)
def test_windows_that_begin_in_the_padding(kernel, channels):
    r = rng_for(8700 + 10 * kernel[0] + kernel[1] + channels)
    x = rand_u8(r, (3, 9, 11, channels))
    # (the largest of no taps is 0: `more` rows and columns of windows that lie wholly past the image, which the oracle does not know)
    for strides, pads, out_hw, more in (((2, 2), (1, 1, 1, 1), (5, 6), 0), ((3, 2), (2, 0, 1, 2), (5, 4), 0), ((2, 2), (1, 1, 1, 1), (5, 6), 3),
                                        ((3, 3), (0, 0, 0, 0), (3, 4), 2)):
        pads = (min(pads[0], kernel[1] - 1), pads[1], min(pads[2], kernel[0] - 1), pads[3])  # (a tap of every window in the image)
        want = np.pad(oracle.maxpool(x, kernel, strides, pads, out_hw=out_hw), ((0, 0), (0, more), (0, more), (0, 0)))
        got = maxpool(x, kernel, strides, (out_hw[0] + more, out_hw[1] + more), pads)[0]
        assert_same(got, want, "max %s %s" % (strides, pads))
    for strides, pads, out_hw in (((2, 2), (1, 1, 1, 1), (5, 6)), ((2, 2), (0, 1, 1, 0), (5, 6)), ((3, 2), (2, 1, 0, 1), (4, 4)),
                                  ((3, 3), (1, 1, 1, 1), (5, 6))):
        for bits in (32, 64):
            want = oracle.avgpool(x, kernel, strides, pads, out_hw, 300, 7, 900, 1, bits)
            assert_same(avgpool(x, kernel, strides, out_hw, pads, 300, 7, 900, 1, bits), want, "average %s %s" % (strides, pads))
