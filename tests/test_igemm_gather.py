"""The activation loads of igemm_kernel at 16 and 32 input channels, walked on the host (tests/host/igemm_gather_walk.cpp)."""
import os
import random
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rows_past_the_last_pixel_load_nothing(tmp_path):
    """Partly filled tiles, padding, taps past the filter: no load in front of the input or behind it."""
    exe = str(tmp_path / "igemm_gather_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "host", "igemm_gather_walk.cpp"), "-o", exe], check=True)
    r = random.Random(1)
    layers = []
    while len(layers) < 400:
        ci, k, s = r.choice([16, 32]), r.choice([(1, 1), (3, 3), (3, 3), (5, 5), (1, 3), (3, 1), (2, 4)]), r.choice([1, 1, 2])
        if k[0] * k[1] + 64 // ci > 32:  # one bit per tap: the launcher's rule
            continue
        pt, pl, h, w = r.randint(0, k[1]), r.randint(0, k[0]), r.randint(k[1], 20), r.randint(k[0], 20)
        ho, wo = (h + 2 * pt - k[1]) // s + 1, (w + 2 * pl - k[0]) // s + 1
        if ho > 0 and wo > 0:
            layers.append((r.choice([1, 2, 5]), h, w, ci, k[0], k[1], pt, pl, s, s, ho, wo, r.choice([128, 256])))
    res = subprocess.run([exe], input="\n".join(" ".join(map(str, l)) for l in layers), stdout=subprocess.PIPE, text=True, timeout=100)
    said = res.stdout.split("\n")[:-1]
    assert res.returncode == 0 and len(said) == len(layers)
    for l, s in zip(layers, said):
        assert s == "ok", "layer %s: %s" % (l, s)
