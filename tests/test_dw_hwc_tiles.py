"""The rows of dw_hwc_kernel walked on the host (tests/host/dw_hwc_walk.cpp): every load of the byte that is meant, every output byte
written once, at its place, for all layers that the kernel takes."""
import os
import random
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rows_on_the_host(tmp_path):
    exe = str(tmp_path / "dw_hwc_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "host", "dw_hwc_walk.cpp"), "-o", exe], check=True)
    r, layers = random.Random(5), []
    for W, S in ((64, 1), (64, 2), (32, 1), (32, 2), (16, 1)):
        nt = 64 // W
        for _ in range(120):
            H = r.randint(1, 70)
            layers.append((r.choice([1, 2, 3, 17, 64]), 16 * nt * r.randint(1, 5), H, W, r.randint(1, (H - 1) // S + 1), S, r.choice([64, 256])))
        # nearly 2^31 bytes of input, and a little more
        rows = (2 ** 31 - 1) // (W * 16 * nt) - 2
        layers.append((1, 16 * nt, rows, W, (rows - 1) // S + 1, S, 256))
        layers.append((1, 16 * nt, rows + 2, W, (rows - 1) // S + 1, S, 256))
    text = "\n".join(" ".join(map(str, l)) for l in layers)
    res = subprocess.run([exe], input=text, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100)
    assert res.returncode == 0, res.stderr
    said = res.stdout.split("\n")[:-1]
    for l, s in zip(layers, said):
        assert s.startswith("ok") or (s == "no" and l[0] * l[1] * l[2] * l[3] + l[3] * l[1] >= 2 ** 31 - 1), "layer %s: %s" % (l, s)
    assert sum(s == "no" for s in said) == 5


def test_bands_are_even(tmp_path):
    """Bands of nearly one height; the rows that a wave takes are few where that leaves no SIMD a second wave, and where many waves share the
    lines of a pixel in a large layer."""
    exe = str(tmp_path / "dw_hwc_walk")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "host", "dw_hwc_walk.cpp"), "-o", exe], check=True)
    cases = [((334, 32, 35, 64, 35, 1, 256), 12), ((334, 32, 19, 64, 19, 1, 256), 8), ((244, 128, 16, 16, 16, 1, 256), 8),
             ((55, 128, 35, 32, 35, 1, 256), 4), ((64, 128, 11, 16, 11, 1, 256), 2), ((64, 16, 64, 64, 64, 1, 256), 4), ((256, 16, 64, 64, 64, 1, 256), 16),
             ((45, 1024, 32, 32, 32, 1, 256), 8), ((22, 512, 64, 64, 32, 2, 256), 8), ((256, 64, 64, 64, 32, 2, 256), 16), ((1, 16, 3, 64, 3, 1, 256), 1)]
    res = subprocess.run([exe], input="\n".join(" ".join(map(str, c[0])) for c in cases), stdout=subprocess.PIPE, text=True, timeout=100)
    for (c, rows), s in zip(cases, res.stdout.split("\n")):
        assert s == "ok %d" % rows, (c, s)
