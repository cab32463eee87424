"""Depthwise layers on the matrix cores (csrc/dw_mfma.h): the shapes where its tiles, masks and tails change."""
import pytest

import oracle
from gpu_helpers import assert_same, depthwise_generic, rand_s8, rand_u8, rng_for
from pulp_nn_amd import PulpNNError

pytestmark = pytest.mark.gpu

GEOMS = [
    # B, CH, H, W, ky, kx, pads, strides(sx,sy)
    (1, 1, 4, 4, 3, 3, (1, 1, 1, 1), (1, 1)),        # 16 bytes of input: one staged chunk is all of it
    (2, 17, 9, 15, 3, 3, (1, 1, 1, 1), (1, 1)),      # one channel in the last block, one column short of a group
    (2, 15, 5, 17, 3, 3, (1, 1, 1, 1), (1, 1)),      # one column past a group
    (1, 20, 33, 33, 3, 3, (1, 1, 1, 1), (2, 2)),     # two MFMAs per block
    (1, 19, 6, 50, 1, 1, (0, 0, 0, 0), (1, 1)),
    (2, 16, 11, 13, 4, 4, (1, 1, 1, 1), (1, 1)),     # four filter columns: all of a dword
    (1, 18, 12, 21, 5, 5, (2, 2, 2, 2), (1, 1)),
    (1, 9, 14, 23, 7, 7, (3, 3, 3, 3), (1, 1)),      # three MFMAs
    (1, 8, 17, 40, 7, 7, (3, 3, 3, 3), (2, 2)),      # five
    (1, 7, 10, 20, 3, 8, (1, 1, 3, 4), (1, 1)),      # the widest filter: two dwords per filter row
    (1, 5, 20, 9, 9, 2, (4, 4, 0, 1), (1, 3)),       # more filter rows than columns, row stride 3
    (1, 2, 1, 14, 2, 1, (3, 3, 5, 5), (1, 1)),       # 14 bytes a plane, rows that all lie in the padding
    (3, 24, 1, 9, 2, 1, (6, 1, 7, 7), (1, 2)),
    (2, 10, 3, 5, 3, 8, (8, 2, 7, 2), (1, 4)),
    (1, 6, 8, 31, 3, 3, (1, 1, 1, 1), (3, 1)),
    (1, 3, 7, 1000, 1, 3, (0, 0, 1, 1), (1, 1)),    # wider than a tile: several tiles along a row
    (600, 16, 6, 340, 3, 3, (1, 1, 1, 111), (1, 1)),  # two column tiles of two rows, the second one narrower
    (400, 33, 5, 336, 3, 3, (1, 1, 0, 90), (1, 1)),
    (1, 2, 200, 18, 3, 3, (1, 1, 1, 1), (1, 1)),     # several bands of rows
    (600, 70, 7, 7, 3, 3, (1, 1, 1, 1), (1, 1)),     # small planes: 64 channels per workgroup, six in the last one
    (520, 128, 5, 9, 3, 3, (0, 0, 1, 1), (1, 1)),
    (1, 4, 6, 10, 12, 10, (5, 6, 4, 5), (1, 1)),     # a filter wider than 8 columns: the byte loop
]


# where the loads of filters, constants and input rows change form
SETUP_GEOMS = [
    (1, 3, 1, 9, 1, 2, (0, 0, 0, 0), (1, 1)),        # 6 bytes of filters: fewer than one load
    (1, 4, 5, 6, 1, 2, (0, 0, 0, 1), (1, 1)),        # 8 bytes: one load
    (2, 3, 6, 7, 3, 1, (1, 1, 0, 0), (1, 1)),        # 9: the last rows are loaded too early
    (1, 21, 40, 8, 17, 1, (8, 8, 0, 0), (1, 1)),     # 68 filter rows in a wave
    (1, 2, 3, 20, 1, 8, (0, 0, 64, 3), (1, 1)),      # rows that begin 64 bytes before the tensor
    (3, 40, 2, 7, 2, 3, (1, 1, 5, 5), (1, 1)),       # 14 bytes a plane, several blocks of channels
    (2, 33, 3, 6, 3, 3, (1, 1, 1, 1), (1, 1)),       # 18 bytes a plane: a chunk reaches over the next one
    (300, 80, 8, 8, 3, 3, (1, 1, 1, 1), (2, 2)),     # 64 channels per workgroup, 16 in the last: one quad for each wave
    (350, 100, 6, 6, 5, 5, (2, 2, 2, 2), (1, 1)),    # ... 36: three quads for each of three waves
]


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("flags", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("geom", GEOMS + SETUP_GEOMS, ids=lambda g: "x".join(map(str, g[:6])) + "s%d%d" % g[7])
def test_depthwise_shapes(geom, flags, bn_bits):
    B, CH, H, W, ky, kx, pads, strides = geom
    relu, bn = flags
    r = rng_for(7100 + 17 * relu + bn + bn_bits + CH)
    x, wt, b = rand_u8(r, (B, CH, H, W)), rand_s8(r, (CH, ky, kx)), rand_s8(r, (CH,))
    if bn_bits == 32:
        k, lam, bshift = r.integers(2 ** 12, 2 ** 14 + 1, CH), r.integers(-2 ** 16, 2 ** 16 + 1, CH), 18
    else:
        k, lam, bshift = r.integers(2 ** 20, 2 ** 24 + 1, CH), r.integers(-2 ** 36, 2 ** 36 + 1, CH), 28
        k[0] = 2 ** 40       # one multiplier past 32 bits: the plain 64-bit form of the requantisation
    shift = bshift if (relu and bn) else ((17 if CH % 2 else 13) if relu else 6)
    want = oracle.depthwise_generic(x, wt, b, k, lam, 900, shift, pads, strides, relu, bn, bn_bits)
    got = depthwise_generic(x, wt, b, k, lam, 900, shift, pads, strides, relu, bn, bn_bits)
    assert_same(got, want, "depthwise %s" % (geom,))


@pytest.mark.parametrize("width, kernel, accepted", [(331, 3, True), (333, 3, False), (340, 3, True), (343, 3, False),
                                                     (198, 5, True), (199, 5, False)])
def test_depthwise_width_limit(width, kernel, accepted):
    """ky rows of 64 channels in 64 KiB of LDS, 4 bytes left of a row: the widest rows taken and the first refused
    (3 x 3 on rows of whole dwords: no bytes beside the row, so 340 is one of the taken)."""
    r = rng_for(7200 + width)
    pad = (kernel // 2,) * 4
    x, wt, b = rand_u8(r, (1, 3, 6, width)), rand_s8(r, (3, kernel, kernel)), rand_s8(r, (3,))
    args = (x, wt, b, None, None, 900, 13, pad, (1, 1), 1, 0, 32)
    if accepted:
        assert_same(depthwise_generic(*args), oracle.depthwise_generic(*args), "width %d" % width)
    else:
        with pytest.raises(PulpNNError) as e:
            depthwise_generic(*args)
        assert e.value.code == 2
