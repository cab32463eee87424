"""conv_rows_kernel against the oracle: filter rows of every length and place in the input, strides, padding on every side, output rows that
are whole units of 16 and 64 pixels or not, channel counts around whole groups, a first and a last byte of the tensor that a fetch must
not pass, every requantisation form."""
import numpy as np
import pytest

import oracle
from gpu_helpers import assert_same, conv, rand_s8, rand_u8, rng_for

pytestmark = pytest.mark.gpu

GEOMS = [  # B, H, W, Ci, Co, (kx, ky), (sx, sy), (t, b, l, r)
    (1, 3, 11, 1, 16, (3, 3), (1, 1), (1, 1, 1, 1)),
    (2, 9, 64, 3, 16, (3, 3), (1, 1), (1, 1, 1, 1)),
    (3, 8, 130, 3, 16, (3, 3), (2, 2), (1, 0, 1, 0)),        # 65 columns
    (2, 12, 128, 3, 16, (3, 3), (2, 2), (1, 1, 1, 1)),       # groups of 64 pixels of a row
    (1, 6, 192, 5, 24, (3, 4), (1, 1), (2, 1, 1, 1)),        # 15-byte rows that start anywhere
    (2, 7, 48, 4, 40, (4, 4), (1, 2), (3, 0, 2, 1)),         # 16-byte rows, 48 columns
    (1, 5, 33, 7, 17, (2, 2), (1, 1), (1, 1, 1, 1)),
    (2, 10, 32, 16, 33, (1, 3), (1, 1), (1, 1, 0, 0)),
    (3, 6, 16, 13, 70, (1, 1), (1, 1), (0, 0, 0, 0)),
    (40, 20, 40, 3, 100, (3, 3), (1, 1), (1, 1, 1, 1)),      # four 16-channel groups a wave, several groups of pixels
    (300, 16, 64, 3, 32, (5, 2), (1, 1), (0, 1, 4, 0)),
]
STORES = [  # channel counts whose pixels are put together before they are stored, batches that end within a group of 64 pixels
    (253, 15, 19, 2, 7, (4, 1), (1, 1), (0, 0, 1, 1)),
    (3, 5, 16, 13, 14, (1, 1), (1, 1), (0, 0, 0, 0)),
    (1, 3, 23, 4, 1, (3, 3), (1, 1), (1, 1, 1, 1)),
    (2, 5, 64, 3, 3, (3, 3), (1, 1), (1, 1, 1, 1)),
    (70, 33, 16, 4, 47, (3, 3), (1, 1), (1, 1, 1, 1)),
    (64, 17, 64, 3, 63, (3, 2), (1, 1), (1, 0, 1, 1)),
    (20, 37, 49, 3, 30, (3, 3), (1, 1), (1, 1, 1, 1)),
    (1, 2, 17, 16, 29, (1, 2), (1, 1), (1, 0, 0, 0)),
    (9, 48, 54, 2, 7, (1, 1), (1, 1), (0, 0, 0, 0)),         # filters of fewer than 16 bytes in all
    (5, 12, 16, 1, 15, (1, 1), (1, 1), (0, 0, 0, 0)),
    (3, 9, 64, 1, 1, (3, 3), (1, 1), (1, 1, 1, 1)),
    (2, 30, 33, 2, 2, (2, 1), (1, 1), (0, 0, 1, 0)),
    (40, 24, 48, 3, 131, (3, 3), (1, 1), (1, 1, 1, 1)),      # more than one block of channels: the last one's tail by dwords
]


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("geom", GEOMS + STORES, ids=lambda g: "x".join(map(str, g[:5])) + "_%dx%d" % g[5])
def test_rows(geom, bn_bits):
    B, H, W, Ci, Co, (kx, ky), strides, pads = geom
    r = rng_for(8800 + Ci + Co)
    x, w, b = rand_u8(r, (B, H, W, Ci)), rand_s8(r, (Co, ky, kx, Ci)), rand_s8(r, (Co,))
    x[0, 0], x[-1, -1] = 255, 255
    k, lam = r.integers(256, 1025, Co), r.integers(-2 ** 16, 2 ** 16 + 1, Co)
    big = k.copy()
    big[Co // 2] = 2 ** 25 if bn_bits == 32 else 2 ** 33
    for kk, shift, relu, bn in ((k, 17, 1, 1), (big, 17, 1, 1), (k, 14, 1, 0), (k, 16, 1, 0), (k, 7, 0, 0)):
        want = oracle.conv(x, w, b, kk, lam, 700, shift, pads, strides, relu, bn, bn_bits)
        assert_same(conv(x, w, b, kk, lam, 700, shift, pads, strides, relu, bn, bn_bits), want, "relu=%d bn=%d shift=%d" % (relu, bn, shift))
