"""The tiles of dw_mfma_kernel walked on the host (tests/host/dw_mfma_walk.cpp): every load inside the input, every output
pixel written once, at its place."""
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("walk") / "dw_mfma_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "host", "dw_mfma_walk.cpp"), "-o", exe], check=True)

    def run(layers):
        text = "\n".join(" ".join(map(str, l)) for l in layers)
        res = subprocess.run([exe], input=text, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
        assert res.returncode == 0, res.stderr
        return res.stdout.split("\n")[:-1]
    return run


def layer(B, CH, H, W, kx, ky, pads, strides, out_hw=None, bn_bytes=4, cus=256):
    """pads: (top, bottom, left, right)."""
    pt, pb, pl, pr = pads
    sx, sy = strides
    ho, wo = out_hw or ((H + pt + pb - ky) // sy + 1, (W + pl + pr - kx) // sx + 1)
    return B, CH, H, W, ho, wo, kx, ky, pt, pl, sx, sy, bn_bytes, cus


def check(walk, layers, taken=True):
    for l, said in zip(layers, walk(layers)):
        assert said.startswith("ok") or (not taken and said == "no"), "layer %s: %s" % (l, said)


def test_usual_layers(walk):
    r = random.Random(1)
    layers = []
    for _ in range(1500):
        k = r.choice([3, 3, 5, 7])
        s = r.choice([1, 1, 2])
        layers.append(layer(r.choice([1, 2, 33, 256]), r.randint(1, 200), r.randint(k, 70), r.randint(16, 70), k, k, (k // 2,) * 4, (s, s),
                            bn_bytes=r.choice([4, 8])))
    check(walk, layers)


def test_narrow_last_column_tile(walk):
    """Several column tiles and several rows per tile: the last tile's rows are shorter, in LDS too."""
    check(walk, [layer(600, 16, 6, 340, 3, 3, (1, 1, 1, 111), (1, 1)), layer(64, 16, 40, 320, 3, 3, (1, 1, 1, 131), (1, 1)),
                 layer(600, 24, 8, 336, 3, 3, (1, 1, 0, 100), (1, 1), bn_bytes=8)])
    assert walk([layer(600, 16, 6, 340, 3, 3, (1, 1, 1, 111), (1, 1))]) == ["ok 3600"]  # two column tiles, two rows each


def test_more_planes_than_an_int_counts(walk):
    """batch x channels past 2^31: 105 GB and 107 GB of input, which the card holds."""
    check(walk, [layer(2097152, 1024, 7, 7, 3, 3, (1, 1, 1, 1), (1, 1)), layer(4300000, 1000, 5, 5, 3, 3, (1, 1, 1, 1), (1, 1))])
