"""The runs of pixels of pw_any_kernel walked on the host (tests/host/pw_any_walk.cpp)."""
import os
import random
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_pixel_in_one_run(tmp_path):
    exe = str(tmp_path / "pw_any_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "host", "pw_any_walk.cpp"), "-o", exe], check=True)
    r = random.Random(1)
    layers = [(r.randint(1, 10 ** r.randint(2, 7)), r.randint(8, 600), r.randint(1, 600), r.choice([4, 8]), 256) for _ in range(2000)]
    # as many pixels as the entry point takes (an int), and a few less
    layers += [(m, n, k, 4, 256) for m in (2 ** 31 - 1, 2 ** 31 - 16, 2 ** 31 - 64, 2 ** 31 - 100, 2 ** 31 - 5000)
               for n, k in ((16, 1), (24, 20), (300, 20))]
    res = subprocess.run([exe], input="\n".join(" ".join(map(str, l)) for l in layers), stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                         text=True, timeout=100)
    said = res.stdout.split("\n")[:-1]
    assert res.returncode == 0, "layer %s: %s" % (layers[len(said)], res.stderr)
    for l, s in zip(layers, said):
        assert s.startswith("ok") or s == "no", "layer %s: %s" % (l, s)
    assert sum(s != "no" for s in said) > 400
