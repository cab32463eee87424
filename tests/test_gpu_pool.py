"""Pooling (csrc/pool.h): windows of one to seven taps a side on each path of channels, partial windows on every side, and
products of the average's requantisation on both sides of 32 bits."""
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
