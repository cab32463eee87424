"""How many taps the pooling kernels load for a window (tests/host/pool_blocks.cpp): few more than it has, in few trips to memory."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_loads_of_a_window(tmp_path):
    exe = str(tmp_path / "pool_blocks")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "host", "pool_blocks.cpp"), "-o", exe], check=True)
    windows = [(kx, ky) for kx in range(1, 33) for ky in range(1, 33)] + [(65535, 1), (1, 65535), (300, 200)]
    text = "\n".join("%d %d" % w for w in windows)
    out = subprocess.run([exe], input=text, stdout=subprocess.PIPE, text=True, timeout=100, check=True).stdout.split("\n")
    for (kx, ky), line in zip(windows, out):
        avg, avg_trips, most, most_trips = map(int, line.split())
        taps, rows_of_four = kx * ky, ky * -(-kx // 4)
        # never more loads and trips, a trip counting as two loads, than with rows of four taps, nor than with whole squares of four
        assert taps <= avg and avg + 2 * avg_trips <= min(6 * rows_of_four, 18 * -(-kx // 4) * -(-ky // 4)), (kx, ky, line)
        # the maximum loads sixteen bytes a tap: at most a third more than there are, up to 3x3 (and 2x2) the whole window
        assert taps <= most and (most <= 1.34 * taps + 1 if max(kx, ky) > 3 else most <= 9), (kx, ky, line)
        assert most_trips == 1 or max(kx, ky) > 3, (kx, ky, line)
