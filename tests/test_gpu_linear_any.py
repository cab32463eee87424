"""Linear layers whose rows are not whole 16-byte chunks (csrc/linear_skinny.h): lengths around a chunk, a K slice and
the parts K is dealt in; neurons and rows around their blocks; operands that start at an odd address."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import assert_same, linear, linear_out_32, nn, rand_s8, rand_u8, rng_for

pytestmark = pytest.mark.gpu

GEOMS = [
    # rows, K, neurons
    (1, 15, 4), (1, 16, 1), (1, 17, 16), (2, 31, 17), (3, 33, 15), (16, 63, 10), (17, 65, 20), (64, 79, 33), (65, 255, 64),
    (130, 257, 19), (256, 1001, 100), (200, 1000, 4093), (64, 4095, 12), (7, 520, 999), (255, 1027, 2999), (257, 40, 24),
]


# the ring of four K slices (a wave's part of K shorter, as long, longer), one to four groups of 16 rows, one, two and four parts of K
RING = [(1, 1024, 20), (17, 1088, 40), (33, 1280, 17), (49, 2560, 36), (64, 4096, 16), (100, 704, 8208), (250, 320, 8224), (40, 1300, 8208)]


@pytest.mark.parametrize("bn_bits", [32, 64])
@pytest.mark.parametrize("geom", GEOMS + RING, ids=lambda g: "x".join(map(str, g)))
def test_linear_any_length(geom, bn_bits):
    M, K, N = geom
    r = rng_for(8300 + K + bn_bits)
    x, w, b = rand_u8(r, (M, K)), rand_s8(r, (N, K)), rand_s8(r, (N,))
    for relu, bn in ((1, 1), (1, 0), (0, 0)):
        if bn_bits == 32:
            k, lam, shift = r.integers(256, 1025, N), r.integers(-2 ** 16, 2 ** 16 + 1, N), 20
        else:
            k, lam, shift = r.integers(2 ** 20, 2 ** 24 + 1, N), r.integers(-2 ** 36, 2 ** 36 + 1, N), 34
        if not (relu and bn):
            shift = (14 if K < 200 else 19) if relu else 8
        want = oracle.linear(x, w, b, k, lam, 700, shift, relu, bn, bn_bits)
        assert_same(linear(x, w, b, k, lam, 700, shift, relu, bn, bn_bits), want, "linear %s relu %d bn %d" % (geom, relu, bn))
    b32 = r.integers(-2 ** 20, 2 ** 20, N).astype(np.int32)
    assert_same(linear_out_32(x, w, b32, bn_bits), oracle.linear_out_32(x, w, b32), "linear_out_32 %s" % (geom,))


@pytest.mark.parametrize("offsets", [(1, 0, 0), (0, 3, 0), (0, 0, 2), (5, 7, 1)], ids=str)
def test_linear_any_address(offsets):
    M, K, N = 20, 64, 48  # whole chunks: only the addresses are odd
    r = rng_for(8400 + sum(offsets))
    x, w, b = rand_u8(r, (M, K)), rand_s8(r, (N, K)), rand_s8(r, (N,))
    xi, wi, out = [torch.zeros(n + 16, dtype=d, device="cuda")[o:o + n] for n, d, o in
                   zip((M * K, N * K, M * N), (torch.uint8, torch.int8, torch.uint8), offsets)]
    xi.copy_(torch.from_numpy(x.reshape(-1)))
    wi.copy_(torch.from_numpy(w.reshape(-1)))
    L = nn(32)
    L.set_batch(M)
    L.pulp_nn_linear(xi, torch.from_numpy(b).cuda(), out, wi, None, None, 700, 14, K, N, 1, 0)
    want = oracle.linear(x, w, b, None, None, 700, 14, 1, 0, 32)
    assert_same(out.cpu().numpy().reshape(M, N), want, "linear at %s" % (offsets,))
