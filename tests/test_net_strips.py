"""The start net's division of images among waves (csrc/trl_strips.h),
compiled for the CPU: every pixel belongs to exactly one strip, and no wave
sums more of a weight gradient in FP32 than an even split of the pixels in
runs of 32 over 1,024 waves gives it, within a quarter and a strip's row."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "nutrlan_amd", "csrc")
SHAPES = [(1, 3, 3), (1, 64, 64), (8, 64, 64), (9, 65, 63), (16, 64, 33), (40, 64, 33), (64, 64, 64), (70, 64, 64),
          (64, 3, 3), (3000, 3, 3), (500, 5, 7), (64, 8, 8), (200, 31, 16), (90, 12, 40), (130, 17, 33), (4, 256, 256),
          (1, 512, 512), (16, 100, 100), (6, 200, 200), (2, 1000, 3), (2, 3, 1000),
          (900, 15, 15), (1500, 11, 11), (10000, 5, 5), (500, 33, 33)]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("strips") / "strips_cover")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, os.path.join(HERE, "strips_cover.cpp"), "-o", out],
                   check=True)
    return out


@pytest.fixture(scope="module")
def counts(exe):
    args = [str(v) for s in SHAPES for v in s]
    out = subprocess.run([exe, *args], capture_output=True, text=True, check=True).stdout.splitlines()
    return [(s, [int(v) for v in line.split()]) for s, line in zip(SHAPES, out)]


def test_gradient_strips(counts):
    for (nimg, h, w), (bad, most, *_) in counts:
        width = -(-w // -(-w // 32))
        even = 32 * -(-(-(-nimg * h * w // 32)) // 1024)
        assert bad == 0, (nimg, h, w)
        assert most <= even + even // 4 + width, (nimg, h, w, most, even)


def test_convolution_strips(counts):
    """Every pixel once, at every height a walk may have; narrow images share
    strips, so that 9 of 16 lanes or more have a pixel (but in the last)."""
    for (nimg, h, w), (_, _, _, bad, neighbours, waves) in counts:
        assert bad == 0 and neighbours == 0, (nimg, h, w)
        if w <= 8:
            assert 9 * waves <= -(-h // 8) * (nimg * w + 16), (nimg, h, w, waves)
