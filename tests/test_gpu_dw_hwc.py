"""dw_hwc_kernel against the oracle: rows of every width and stride it takes, heights around the rows a wave takes, several channel
groups, batches that leave the last workgroup partly empty, both requantisation forms of every mode."""
import numpy as np
import pytest

import oracle
from gpu_helpers import assert_same, depthwise_hwc, rand_s8, rand_u8, rng_for

pytestmark = pytest.mark.gpu

GEOMS = [  # B, CH, H, W, stride
    (4, 16, 1, 64, 1), (4, 48, 19, 64, 1), (256, 16, 21, 64, 1), (4, 16, 2, 64, 2), (12, 80, 35, 64, 2), (256, 16, 38, 64, 2),
    (2, 32, 3, 32, 1), (2, 96, 33, 32, 1), (130, 64, 18, 32, 1), (2, 32, 1, 32, 2), (6, 160, 37, 32, 2), (258, 32, 30, 32, 2),
    (1, 64, 1, 16, 1), (3, 192, 17, 16, 1), (257, 64, 20, 16, 1),
]
EVEN = [  # several bands a plane, the last one shorter; few rows per wave; many channel groups
    (256, 16, 35, 64, 1), (200, 32, 19, 64, 1), (130, 64, 35, 32, 2), (24, 128, 35, 64, 1), (24, 128, 37, 64, 2), (40, 128, 18, 32, 1), (244, 128, 16, 16, 1),
    (64, 192, 7, 16, 1),
]


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("geom", GEOMS + EVEN, ids=lambda g: "x".join(map(str, g[:4])) + "s%d" % g[4])
def test_rows(geom, bn_bits):
    B, CH, H, W, S = geom
    r = rng_for(9100 + CH + H)
    x, wt, b = rand_u8(r, (B, H, W, CH)), rand_s8(r, (CH, 3, 3)), rand_s8(r, (CH,))
    x[:, 0] = 255      # the rows and columns next to the padding at the largest value
    x[:, :, -1] = 255
    x_chw = np.ascontiguousarray(x.transpose(0, 3, 1, 2))
    if geom in EVEN:   # (larger ones: the first and the last images)
        pick = sorted({0, 1, B - 1})
    else:
        pick = list(range(B))
    x_chw = x_chw[pick]
    small = (r.integers(256, 1025, CH), r.integers(-2 ** 16, 2 ** 16 + 1, CH), 17)
    large = (small[0].copy(), small[1], 17)
    large[0][CH // 2] = 2 ** 25 if bn_bits == 32 else 2 ** 33     # past the fast multiplier: 24 or 32 bits
    for (k, lam, shift), relu, bn in ((small, 1, 1), (large, 1, 1), ((small[0], small[1], 14), 1, 0), ((small[0], small[1], 16), 1, 0),
                                      ((small[0], small[1], 7), 0, 0)):
        want = oracle.depthwise_generic(x_chw, wt, b, k, lam, 700, shift, (1, 1, 1, 1), (S, S), relu, bn, bn_bits)
        assert_same(depthwise_hwc(x, wt, b, k, lam, 700, shift, S, relu, bn, bn_bits)[pick], want, "relu=%d bn=%d shift=%d" % (relu, bn, shift))


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("geom", [(68, 128, 64, 64, 1), (130, 128, 64, 64, 2), (700, 128, 13, 64, 2)], ids=lambda g: "x".join(map(str, g[:4])) + "s%d" % g[4])
def test_large_rows_of_many_channels(geom, bn_bits):
    """Layers whose size takes them to the other kernel: the same bytes as in two halves, which do not."""
    B, CH, H, W, S = geom
    r = rng_for(9300 + H)
    x, wt, b = rand_u8(r, (B, H, W, CH)), rand_s8(r, (CH, 3, 3)), rand_s8(r, (CH,))
    k, lam = r.integers(256, 1025, CH), r.integers(-2 ** 16, 2 ** 16 + 1, CH)
    for shift, relu, bn in ((17, 1, 1), (14, 1, 0), (7, 0, 0)):
        got = depthwise_hwc(x, wt, b, k, lam, 700, shift, S, relu, bn, bn_bits)
        for part in (slice(0, B // 2), slice(B // 2, B)):
            assert_same(got[part], depthwise_hwc(x[part], wt, b, k, lam, 700, shift, S, relu, bn, bn_bits), "relu=%d bn=%d shift=%d" % (relu, bn, shift))
