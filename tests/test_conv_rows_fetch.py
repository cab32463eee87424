"""The fetches of conv_rows_kernel walked on the host (tests/host/conv_rows_walk.cpp): no byte outside the input, every byte of a filter row in
its place, for strides, paddings and channel counts of the whole range."""
import os
import random
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_fetches_on_the_host(tmp_path):
    exe = str(tmp_path / "conv_rows_walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "host", "conv_rows_walk.cpp"), "-o", exe], check=True)
    r, layers = random.Random(3), []
    for _ in range(900):
        kx = r.choice([1, 1, 2, 3, 3, 3, 4, 5, 7])
        ky, Ci = r.choice([1, 2, 3, 3, 4]), r.randint(1, max(1, 16 // kx))
        sx, sy = r.choice([1, 1, 2, 3]), r.choice([1, 1, 2, 5])
        pl, pt = r.randint(0, kx), r.randint(0, ky)
        Wo, Ho = r.choice([16, 32, 64, 128] + [r.randint(1, 70)] * 4), r.randint(1, 6)
        W = max(1, (Wo - 1) * sx + kx - pl - r.randint(0, 2 * pl))
        H = max(1, (Ho - 1) * sy + ky - pt - r.randint(0, pt))
        layers.append((r.choice([1, 1, 2, 3]), H, W, Ci, kx, ky, pt, pl, sx, sy, Ho, Wo, 16))
    layers.append((43691, 128, 128, 3, 3, 3, 1, 1, 2, 2, 64, 64, 16))     # past 2^31 bytes of input
    res = subprocess.run([exe], input="\n".join(" ".join(map(str, l)) for l in layers), stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                         timeout=100)
    said = res.stdout.split("\n")[:-1]
    for l, s in zip(layers, said):
        assert s == "ok" or (s == "no" and (l[0] * l[1] * l[2] * l[3] < 32 or l[0] == 43691 or 16 * l[3] * l[4] * l[5] < 16)), "layer %s: %s" % (l, s)
    assert res.returncode == 0, res.stderr
    assert len(said) == len(layers) and said.count("ok") > 800
