"""Which of two kernels a size gets (csrc/launch_rules.h), pinned on both sides of every line at sizes where both were
timed: the one named is the faster one there."""
import subprocess

import build_cpp


def _ask(lines):
    binary = build_cpp.build("host_launch_rules")
    out = subprocess.run([binary], input="\n".join(lines), text=True, capture_output=True, check=True).stdout
    return [int(x) for x in out.split()]


def test_fwgemm_takes_the_faster_kernel():
    one, tile, half = 1, 2, 3
    cases = [  # f64, k-contiguous image of A at hand, n, kernel
        (0, 0, 1000, one), (0, 0, 1152, one), (0, 0, 1408, one), (0, 0, 1536, tile), (0, 0, 2048, tile),
        (0, 1, 896, one), (0, 1, 1000, one), (0, 1, 1024, one), (0, 1, 1100, one), (0, 1, 1152, tile), (0, 1, 2100, tile),
        (1, 0, 800, one), (1, 0, 900, one), (1, 0, 1000, half), (1, 0, 1280, half), (1, 0, 1792, half),
        (1, 1, 700, one), (1, 1, 768, one), (1, 1, 800, half), (1, 1, 1024, half), (1, 1, 1408, half), (1, 1, 1536, tile), (1, 1, 2048, tile)]
    got = _ask(["fwgemm %d %d %d %d" % (f64, image, n, n) for f64, image, n, _ in cases])
    assert got == [kernel for *_, kernel in cases]
