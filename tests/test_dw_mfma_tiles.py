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


def layer(B, CH, H, W, kx, ky, pads, strides, out_hw=None, cus=256):
    """pads: (top, bottom, left, right)."""
    pt, pb, pl, pr = pads
    sx, sy = strides
    ho, wo = out_hw or ((H + pt + pb - ky) // sy + 1, (W + pl + pr - kx) // sx + 1)
    return B, CH, H, W, ho, wo, kx, ky, pt, pl, sx, sy, cus


def check(walk, layers, taken=True):
    for l, said in zip(layers, walk(layers)):
        assert said.startswith("ok") or (not taken and said == "no"), "layer %s: %s" % (l, said)


def test_usual_layers(walk):
    r = random.Random(1)
    layers = []
    for _ in range(1500):
        k = r.choice([3, 3, 5, 7])
        s = r.choice([1, 1, 2])
        layers.append(layer(r.choice([1, 2, 33, 256]), r.randint(1, 200), r.randint(k, 70), r.randint(16, 70), k, k, (k // 2,) * 4, (s, s)))
    check(walk, layers)


def test_channels_that_do_not_exist(walk):
    """The last block of channels is short: what a pass asks for beyond them is out of range by the lane's own offset."""
    check(walk, [layer(2, 17, 20, 20, 3, 3, (1, 1, 1, 1), (1, 1)), layer(5, 18, 60, 61, 5, 5, (2, 2, 2, 2), (1, 1)),
                 layer(2, 17, 200, 200, 3, 3, (1, 1, 1, 1), (1, 1)), layer(1100, 65, 7, 7, 3, 3, (1, 1, 1, 1), (1, 1))])


def test_64_channels_a_workgroup_where_planes_are_whole(walk):
    wide = [layer(256, 512, 7, 7, 3, 3, (1, 1, 1, 1), (1, 1)), layer(256, 256, 7, 7, 5, 5, (2, 2, 2, 2), (1, 1)),
            layer(700, 130, 4, 4, 3, 3, (1, 1, 1, 1), (1, 1)), layer(1024, 64, 8, 8, 3, 3, (1, 1, 1, 1), (1, 1))]
    not_wide = [layer(256, 256, 13, 13, 3, 3, (1, 1, 1, 1), (2, 2)), layer(256, 256, 7, 7, 7, 7, (3, 3, 3, 3), (1, 1)),   # cut in bands
                layer(1023, 64, 8, 8, 3, 3, (1, 1, 1, 1), (1, 1)), layer(1024, 64, 8, 9, 3, 3, (1, 1, 1, 1), (1, 1))]
    assert all(s.startswith("ok") and s.endswith("wide") for s in walk(wide))
    assert all(s.startswith("ok") and not s.endswith("wide") for s in walk(not_wide))


def test_narrow_last_column_tile(walk):
    """Several column tiles and several rows per tile: the last tile's rows are shorter, in LDS too."""
    check(walk, [layer(600, 16, 6, 340, 3, 3, (1, 1, 1, 111), (1, 1)), layer(64, 16, 40, 320, 3, 3, (1, 1, 1, 131), (1, 1)),
                 layer(600, 24, 8, 336, 3, 3, (1, 1, 0, 100), (1, 1))])
    assert walk([layer(600, 16, 6, 340, 3, 3, (1, 1, 1, 111), (1, 1))]) == ["ok 3600"]  # two column tiles, two rows each


def test_more_planes_than_an_int_counts(walk):
    """batch x channels past 2^31: 105 GB and 107 GB of input, which the card holds."""
    check(walk, [layer(2097152, 1024, 7, 7, 3, 3, (1, 1, 1, 1), (1, 1)), layer(4300000, 1000, 5, 5, 3, 3, (1, 1, 1, 1), (1, 1))])


def test_tiny_planes_with_wide_padding(walk):
    """Planes of fewer than 16 bytes: a row outside the image must not load past the last one."""
    layers = [layer(1, 2, 1, 14, 1, 2, (3, 3, 5, 5), (1, 1)), layer(2, 10, 3, 5, 8, 3, (8, 2, 7, 2), (1, 4)),
              layer(5, 24, 1, 9, 1, 2, (6, 1, 62, 7), (1, 2)), layer(2, 3, 1, 4, 5, 2, (5, 5, 25, 8), (3, 4))]
    r = random.Random(2)
    while len(layers) < 8000:
        H, W, kx, ky = r.choice([1, 1, 2, 2, 3, 4, 5, 8]), r.randint(1, 20), r.randint(1, 8), r.randint(1, 8)
        pads = [r.randint(0, 8) for _ in range(4)]
        if r.random() < 0.2:
            pads[r.choice([0, 2])] = r.randint(0, 64)
        if H + pads[0] + pads[1] >= ky and W + pads[2] + pads[3] >= kx:
            layers.append(layer(r.choice([1, 2, 5]), r.randint(1, 40), H, W, kx, ky, pads, (r.randint(1, 4), r.randint(1, 5))))
    check(walk, layers, taken=False)


def test_row_stride_far_past_the_image(walk):
    """Output rows whose input rows reach further than an int counts: the tile is sized by what it would take."""
    r = random.Random(3)
    layers = [layer(1, 16, 8, 16, 3, 3, (1, 1, 1, 1), (1, 60000), out_hw=(2000, 16))]
    for _ in range(300):
        layers.append(layer(r.choice([1, 4]), r.randint(1, 70), r.randint(1, 60), r.randint(16, 60), 3, 3, (1, 1, 1, 1),
                            (r.choice([1, 2]), r.randint(1, 65535)), out_hw=(r.choice([100, 1000, 30000]) + r.randint(0, 99), r.randint(1, 80))))
    check(walk, layers)
