"""Convolution and pointwise layers of any channel count (csrc/conv_band.h, csrc/pw_any.h): the shapes where their
tiles, tails and blocks of channels change."""
import pytest

import oracle
from gpu_helpers import assert_same, conv, rand_s8, rand_u8, rng_for

pytestmark = pytest.mark.gpu

CONV = [
    # B, H, W, Ci, Co, ky, kx, pads(t,b,l,r), strides(sx,sy)
    (1, 4, 5, 1, 40, 5, 5, (2, 2, 2, 2), (1, 1)),      # one channel: the first pixels' chunk starts before the tensor
    (2, 6, 7, 2, 33, 3, 3, (1, 1, 1, 1), (1, 1)),
    (1, 9, 11, 15, 17, 3, 3, (1, 1, 1, 1), (2, 2)),    # one byte short of a chunk; two waves along the channels
    (2, 8, 8, 17, 16, 3, 3, (1, 0, 1, 0), (1, 1)),     # one byte past a chunk; one wave along the channels
    (1, 5, 40, 24, 65, 3, 3, (1, 1, 1, 1), (1, 1)),    # one channel past a block of 64: two groups per wave
    (1, 6, 9, 40, 130, 3, 3, (1, 1, 1, 1), (1, 1)),    # four groups per wave
    (1, 6, 9, 40, 300, 2, 3, (0, 1, 1, 1), (1, 2)),    # two blocks of channels
    (1, 3, 700, 20, 24, 3, 3, (1, 1, 1, 1), (1, 1)),   # a row of several tiles, the last one shorter
    (300, 9, 13, 24, 48, 3, 3, (1, 1, 1, 1), (1, 1)),  # enough workgroups for 128 pixels each
    (2, 7, 9, 250, 20, 5, 5, (2, 2, 2, 2), (1, 1)),    # K = 6250: several rounds of weight prefetch
    (1, 20, 17, 144, 35, 3, 3, (1, 1, 1, 1), (1, 1)),  # whole chunks, few output channels
]
# where the band kernel's groups of weights, its passes over the input and its tiles change form
BAND = [
    (2, 10, 19, 112, 32, 3, 3, (1, 1, 1, 1), (1, 1)),   # few workgroups, 16 K steps: groups of four
    (1, 12, 20, 250, 16, 3, 3, (1, 1, 1, 1), (2, 2)),   # ... an odd number of groups, one wave along the channels
    (1, 3, 4, 4100, 5, 2, 2, (0, 0, 0, 0), (1, 1)),     # 257 chunks a pixel: two rounds of 256
    (3, 9, 6, 3, 70, 7, 7, (3, 3, 3, 3), (1, 1)),       # three channels, 13 K steps: the first 16 chunks of channel 0 in several groups
    (1, 6, 8, 1, 140, 4, 5, (2, 1, 2, 2), (1, 1)),      # ... and one channel with four groups of 16 a wave
    (260, 6, 7, 24, 100, 3, 3, (1, 1, 1, 1), (1, 1)),   # two groups a wave, eight of pixels
    (40, 21, 26, 8, 150, 3, 3, (1, 1, 1, 1), (1, 1)),   # four and four
    (1, 5, 150, 256, 20, 5, 5, (2, 2, 2, 2), (2, 1)),   # a tile that LDS holds part of a row for
    (10, 55, 63, 178, 33, 5, 5, (2, 2, 2, 2), (2, 2)),  # weights one step at a time: two workgroups a compute unit
    (21, 13, 53, 256, 17, 5, 5, (2, 2, 2, 2), (1, 1)),  # halves of rows, the second one shorter
]
# small layers of the tiled kernel: nine K slices at a time, taps outside the image on every side
TILED = [
    (1, 9, 11, 64, 40, 3, 3, (1, 1, 1, 1), (1, 1)),     # nine slices
    (1, 8, 9, 64, 72, 2, 5, (1, 0, 2, 2), (1, 1)),      # ten
    (2, 7, 8, 128, 70, 3, 3, (1, 1, 1, 1), (2, 2)),     # eighteen
    (1, 6, 7, 192, 100, 3, 3, (2, 1, 0, 2), (1, 2)),    # three times nine, two rows of padding
    (1, 4, 5, 64, 48, 5, 6, (4, 4, 5, 5), (1, 1)),      # a window larger than the image
    (2, 5, 6, 64, 40, 1, 1, (1, 1, 2, 1), (1, 1)),      # one tap, and pixels that lie in the padding
    (2, 6, 5, 32, 70, 1, 1, (1, 2, 1, 1), (2, 1)),
    (1, 7, 6, 16, 36, 3, 5, (1, 1, 2, 2), (1, 1)),      # four taps a slice
]
POINTWISE = [
    # B, H, W, Ci, Co
    (40, 33, 31, 8, 16), (40, 33, 31, 15, 17), (40, 33, 31, 17, 31), (30, 32, 33, 63, 66), (30, 32, 33, 65, 130),
    (30, 32, 33, 130, 255), (24, 33, 33, 257, 64), (24, 33, 33, 500, 100), (24, 33, 33, 512, 260), (40, 32, 32, 48, 424),
    (9, 29, 31, 72, 20), (3, 9, 7, 9, 5), (1, 1, 1, 20, 24), (2, 5, 5, 600, 30),
    (75, 30, 31, 320, 8),  # (band kernel: weights a step at a time)
    # several pixels of 16 or 32 channels in a column of the matrix cores: whole loads of 64 or 32 pixels, a partial last one, and below the line
    (64, 64, 64, 16, 16), (70, 61, 63, 16, 16), (65, 64, 64, 16, 32), (67, 63, 63, 16, 32), (130, 32, 64, 32, 64), (131, 31, 67, 32, 64),
    (63, 64, 65, 16, 32), (41, 29, 31, 32, 64),
]


def _requant(r, n, bn_bits, relu, bn, K):
    if bn_bits == 32:
        k, lam, shift = r.integers(256, 1025, n), r.integers(-2 ** 16, 2 ** 16 + 1, n), 20
    else:
        k, lam, shift = r.integers(2 ** 20, 2 ** 24 + 1, n), r.integers(-2 ** 36, 2 ** 36 + 1, n), 34
        k[0] = 2 ** 40                     # one multiplier past 32 bits
    if not (relu and bn):
        shift = (14 if K < 200 else 19) if relu == 1 else 8
    return k, lam, shift


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("flags", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("geom", CONV + BAND + TILED, ids=lambda g: "x".join(map(str, g[:7])))
def test_conv_any_channels(geom, flags, bn_bits):
    B, H, W, Ci, Co, ky, kx, pads, strides = geom
    relu, bn = flags
    r = rng_for(8100 + 17 * relu + bn + bn_bits + Ci)
    x, w, b = rand_u8(r, (B, H, W, Ci)), rand_s8(r, (Co, ky, kx, Ci)), rand_s8(r, (Co,))
    k, lam, shift = _requant(r, Co, bn_bits, relu, bn, ky * kx * Ci)
    want = oracle.conv(x, w, b, k, lam, 700, shift, pads, strides, relu, bn, bn_bits)
    assert_same(conv(x, w, b, k, lam, 700, shift, pads, strides, relu, bn, bn_bits), want, "conv %s" % (geom,))


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("flags", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("geom", POINTWISE, ids=lambda g: "x".join(map(str, g)))
def test_pointwise_any_channels(geom, flags, bn_bits):
    B, H, W, Ci, Co = geom
    relu, bn = flags
    r = rng_for(8200 + 17 * relu + bn + bn_bits + Ci)
    x, w, b = rand_u8(r, (B, H, W, Ci)), rand_s8(r, (Co, 1, 1, Ci)), rand_s8(r, (Co,))
    k, lam, shift = _requant(r, Co, bn_bits, relu, bn, Ci)
    want = oracle.pointwise(x, w, b, k, lam, 700, shift, relu, bn, bn_bits)
    got = conv(x, w, b, k, lam, 700, shift, (0, 0, 0, 0), (1, 1), relu, bn, bn_bits, out_hw=(H, W),
               fn="pulp_nn_pointwise_HoWo_parallel")
    assert_same(got, want, "pointwise %s" % (geom,))
