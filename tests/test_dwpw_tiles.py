"""The tiles of the depthwise + pointwise kernels walked on the host (tests/host/dwpw_walk.cpp): a tile for every shape that the entry points
take; for a sample of them, every operand the right pixel's, every activation written once."""
import os
import random
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_tiles_on_the_host(tmp_path):
    exe = str(tmp_path / "dwpw_walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "host", "dwpw_walk.cpp"), "-o", exe], check=True)
    r, blocks = random.Random(11), []
    for W in (64, 32, 16, 8, 4):
        for S in (1, 2):
            for C in [16, 32] + [64 * n for n in (1, 2, 3, 4, 5, 6, 8, 11, 16)]:
                for chained in ((0, 1, 1) if S == 1 else (0,)):
                    for _ in range(3):
                        H = r.choice([4, 8, 8, 16, 16, 24, 32, 40, 64]) - (r.randint(0, 1) if S == 2 else 0)
                        Co = C if chained else 16 * r.choice([1, 2, 3, 5, 8, 16, 32, 64, 100])
                        blocks.append((r.choice([1, 2, 4, 7, 60, 64, 256]), C, H, W, Co, S, chained, r.choice([4, 8]), r.choice([64, 256])))
    every = subprocess.run([exe], input="every", stdout=subprocess.PIPE, text=True, timeout=110).stdout.strip()
    assert every.isdigit() and int(every) > 5000000, every
    # (more images and channels than a tile has room for at once, and slabs of different widths)
    blocks += [(b, C, H, W, Co, S, 0, bn, 256) for W, H, S in ((4, 4, 1), (8, 8, 1), (8, 8, 2), (16, 16, 2), (16, 3, 2), (64, 20, 1)) for C in (64, 192, 448, 704, 1024)
               for b in (40, 300, 513, 1025) for Co in (48, 512) for bn in (4, 8) if b * H * W * C < 4e7]
    res = subprocess.run([exe], input="\n".join(" ".join(map(str, b)) for b in blocks), stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                         timeout=110)
    said = res.stdout.split("\n")[:-1]
    for b, s in zip(blocks, said):
        assert s.startswith("ok") or s == "no", "block %s: %s" % (b, s)
    assert res.returncode == 0, res.stderr
    # (the line of the kernel with five waves a SIMD: a second workgroup that LDS holds and that can begin beside the pointwise stage of the first)
    lean = [(268, 256, 16, 16, 64, 1), (300, 192, 16, 16, 64, 1), (500, 128, 16, 16, 32, 1), (64, 128, 32, 32, 32, 1)]
    not_lean = [(64, 256, 16, 16, 64, 1), (268, 256, 16, 16, 128, 1), (268, 128, 16, 16, 64, 1), (64, 256, 8, 8, 512, 2), (268, 64, 16, 16, 64, 1)]
    text = "\n".join("%d %d %d %d %d %d 0 4 256" % b for b in lean + not_lean)
    line = subprocess.run([exe], input=text, stdout=subprocess.PIPE, text=True, timeout=110).stdout.split("\n")[:-1]
    assert [s.endswith("lean") for s in line] == [True] * len(lean) + [False] * len(not_lean), line
    taken = [b for b, s in zip(blocks, said) if s != "no"]
    assert len(said) == len(blocks) and len(taken) > 200 and sum(b[6] for b in taken) > 30
