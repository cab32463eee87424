"""The tile shapes of conv_band_kernel walked on the host (tests/host/conv_band_walk.cpp): everything a tile stages and reads
inside the LDS it asks for, every output computed once."""
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("walk") / "conv_band_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "host", "conv_band_walk.cpp"), "-o", exe], check=True)

    def run(layers):
        text = "\n".join(" ".join(map(str, l)) for l in layers)
        res = subprocess.run([exe], input=text, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
        said = res.stdout.split("\n")[:-1]
        assert res.returncode == 0, "layer %s: %s" % (layers[len(said)], res.stderr)
        for l, s in zip(layers, said):
            assert s.startswith("ok") or s == "no", "layer %s: %s" % (l, s)
        return said
    return run


def layer(B, H, W, Ci, Ho, Wo, N, kx, ky, pt=0, pl=0, sx=1, sy=1, bn_bytes=4, cus=256):
    return B, H, W, Ci, Ho, Wo, N, kx, ky, pt, pl, sx, sy, bn_bytes, cus


def test_usual_layers(walk):
    r = random.Random(1)
    layers = []
    for _ in range(4000):
        k, s, H, W = r.choice([1, 3, 3, 5, 7]), r.choice([1, 1, 2]), r.randint(7, 70), r.randint(7, 70)
        layers.append(layer(r.choice([1, 2, 33, 256]), H, W, r.randint(3, 300), (H - 1) // s + 1, (W - 1) // s + 1, r.randint(1, 300), k, k,
                            k // 2, k // 2, s, s, bn_bytes=r.choice([4, 8])))
    said = walk(layers)
    assert sum(s != "no" for s in said) > 3500


def test_odd_channel_counts_up_to_128_outputs(walk):
    """The line between this kernel and the tiled one, from both sides."""
    def conv(B, H, W, Ci, N, k, s, bn_bytes=4):
        return layer(B, H, W, Ci, (H + k // 2 * 2 - k) // s + 1, (W + k // 2 * 2 - k) // s + 1, N, k, k, k // 2, k // 2, s, s, bn_bytes=bn_bytes)
    band = [conv(146, 12, 12, 112, 71, 3, 1), conv(177, 27, 8, 176, 120, 3, 1), conv(101, 48, 18, 96, 100, 3, 2), conv(2, 37, 30, 80, 65, 7, 2, 8),
            conv(48, 9, 9, 96, 128, 3, 1), conv(40, 32, 31, 208, 128, 3, 2)]
    tiled = [conv(9, 41, 54, 48, 72, 2, 1), conv(119, 20, 53, 176, 112, 3, 2, 8), conv(182, 24, 48, 176, 96, 3, 2), conv(39, 63, 21, 96, 96, 3, 2),
             conv(92, 10, 17, 96, 120, 3, 1, 8), conv(54, 42, 31, 48, 96, 3, 1), conv(2, 20, 20, 208, 100, 5, 1), conv(8, 16, 16, 96, 128, 1, 1),
             conv(8, 16, 16, 128, 128, 3, 1), conv(8, 16, 16, 96, 129, 3, 1), conv(19, 62, 50, 240, 120, 2, 2),
             conv(133, 16, 28, 176, 128, 3, 1), conv(119, 33, 15, 48, 128, 3, 1)]
    assert all(s.endswith("odd") for s in walk(band))
    assert not any(s.endswith("odd") for s in walk(tiled))


def _conv(B, H, W, Ci, N, k, s, bn_bytes=4):
    return layer(B, H, W, Ci, (H + k // 2 * 2 - k) // s + 1, (W + k // 2 * 2 - k) // s + 1, N, k, k, k // 2, k // 2, s, s, bn_bytes=bn_bytes)


def test_room_for_a_second_workgroup(walk):
    """More workgroups than compute units, of which LDS would hold one with two steps of weights: one step, or halves of rows."""
    one_step = [_conv(10, 55, 63, 178, 33, 5, 2), _conv(16, 55, 64, 178, 64, 5, 2, 8), _conv(73, 14, 54, 224, 32, 5, 2, 8)]
    halves = [_conv(21, 13, 53, 256, 17, 5, 1), _conv(28, 13, 53, 256, 32, 5, 1, 8)]
    whole = [_conv(36, 25, 57, 250, 48, 5, 2), _conv(29, 15, 51, 224, 32, 7, 1)]  # (halves would come out even)
    for l, said in zip(one_step + halves + whole, walk(one_step + halves + whole)):
        lds, tiles = map(int, said.split()[1:3])
        rows = l[0] * l[4]
        assert (lds <= 80 * 1024) == (l not in whole) and tiles == (2 * rows if l in halves else rows), l


def test_33_to_64_outputs(walk):
    """The line between this kernel and the tiled one, from both sides."""
    band = [_conv(32, 42, 61, 80, 40, 3, 1), _conv(94, 48, 39, 144, 63, 3, 2), _conv(47, 39, 45, 240, 40, 5, 2), _conv(48, 11, 50, 224, 40, 7, 2), _conv(163, 15, 54, 48, 40, 3, 1),
            _conv(36, 41, 32, 144, 48, 3, 2)]
    tiled = [_conv(144, 41, 32, 144, 48, 3, 2), _conv(183, 36, 44, 160, 39, 3, 2, 8), _conv(144, 12, 61, 224, 48, 5, 2, 8), _conv(28, 38, 57, 224, 48, 7, 2)]
    assert all(s.endswith("odd") for s in walk(band))
    assert not any(s.endswith("odd") for s in walk(tiled))


def test_lds_past_an_int(walk):
    """Strides and filters whose staged input would take more bytes than an int counts: not taken, or in tiles that fit."""
    layers = [layer(1, 60, 60, 57, 15292, 50, 6, 4, 1, sx=34257, sy=35775), layer(1, 60, 60, 53, 11955, 1, 10, 4, 2, sx=1, sy=37077),
              layer(1, 60, 60, 19, 50314, 6, 2, 2, 5, sx=3, sy=63415), layer(1, 500, 500, 12, 6, 38, 77, 1974, 474, sx=4, sy=62959)]
    r = random.Random(2)
    for _ in range(4000):
        big = r.random() < 0.3
        kx, ky = (r.randint(1, 9000), r.randint(1, 9000)) if big else (r.randint(1, 5), r.randint(1, 5))
        layers.append(layer(r.choice([1, 3]), r.randint(1, 500), r.randint(1, 500), r.randint(1, 60), r.randint(1, 65535), r.randint(1, 65535),
                            r.randint(1, 100), kx, ky, 1, 1, r.randint(1, 65535), r.randint(1, 65535)))
    walk(layers)


def test_pointwise_up_to_the_largest_batch(walk):
    """As many pixels as the entry point takes (an int), and a few less."""
    walk([layer(m, 1, 1, 20, 1, 1, 24, 1, 1) for m in (2 ** 31 - 1, 2 ** 31 - 16, 2 ** 31 - 600, 2 ** 31 - 5000, 65535 * 32767)])
