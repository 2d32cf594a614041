"""The pixel around which a deep frame without rebasing places its next reference: the
flagged one nearest the centroid, the first in row order of those as near."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pick") / "glitch_pick")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-ffp-contract=off",
                    "-fsanitize=address,undefined", "-fno-sanitize-recover",
                    os.path.join(ROOT, "tests", "emulate", "glitch_pick.cpp"), "-o", exe], check=True)

    def run(flags):
        out = subprocess.run([exe, str(flags.shape[1]), str(flags.shape[0])], input=flags.tobytes(),
                             check=True, stdout=subprocess.PIPE)
        return [int(x) for x in out.stdout.split()]
    return run


def expected(flags):
    ys, xs = np.nonzero(flags)
    if len(xs) == 0:
        return [0]
    # whole numbers: their sums are exact in any order
    cx, cy = float(xs.sum()) / len(xs), float(ys.sum()) / len(ys)
    d2 = (xs - cx) * (xs - cx) + (ys - cy) * (ys - cy)
    k = int(np.argmin(d2))
    return [len(xs), int(xs[k]), int(ys[k])]


@pytest.mark.parametrize("density", [0.0, 0.002, 0.1, 1.0])
@pytest.mark.parametrize("width,height", [(1, 1), (7, 3), (8, 5), (9, 4), (15, 2), (16, 16), (23, 31), (640, 37)])
def test_same_pixel_as_one_flag_at_a_time(pick, width, height, density):
    rng = np.random.default_rng(width * 100 + height)
    for k in range(3):
        flags = (rng.random((height, width)) < density).astype(np.uint8)
        if k == 2:
            flags[-1, -1] = 1 + int(rng.integers(0, 255))
        assert pick(flags) == expected(flags)
