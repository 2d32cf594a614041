"""The perturbation kernel's rebasing blocks, modelled on the CPU, against the oracle.

tests/emulate/perturb_rebasing.cpp takes the blocks in which each lane restarts the
reference on its own, the escapes replayed from their block's start and the cycle test,
on 8x8-pixel waves of 1920x1080 frames, and compares count, state and |z|^2 with the
oracle's checked loop bit for bit; it also finds reads outside the orbit.  Frames: few
rebases (1e-20), frequent ones (1e-10, width 1), much interior (1e-6, 0.5), references
of 5 and 7 steps, and iteration limits around a block's length.
"""
import os
import subprocess

import pytest

from conftest import ROOT

CENTRE = ("-0.743643887037151", "0.131825904205330")
CASES = [
    (32, CENTRE, "1e-6", 30000, 12), (64, CENTRE, "1e-6", 30000, 8), (32, CENTRE, "1e-10", 50000, 12),
    (64, CENTRE, "1e-10", 50000, 12), (64, CENTRE, "1e-20", 50000, 6), (32, CENTRE, "1.0", 2000, 12),
    (64, ("-0.25", "0.125"), "1.0", 2000, 12), (32, ("0.5", "0.0"), "1e-3", 2000, 12),
    (64, ("0.7", "0.3"), "0.01", 2000, 12), (64, ("-1.0", "0.0"), "0.5", 700, 12),
    (32, ("0.0", "0.0"), "0.5", 3001, 12), (64, CENTRE, "1e-3", 31, 4), (32, CENTRE, "1e-3", 32, 4),
    (64, CENTRE, "1e-3", 33, 4), (32, CENTRE, "1e-3", 1, 4),
]


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = tmp_path_factory.mktemp("model") / "perturb_rebasing"
    oracle = os.path.join(ROOT, "oracle")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wextra",
           os.path.join(ROOT, "tests", "emulate", "perturb_rebasing.cpp"), "-o", str(exe),
           f"-L{oracle}", "-loracle", f"-Wl,-rpath,{oracle}"]
    build = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if build.returncode != 0:
        pytest.fail(build.stdout[-4000:])
    return str(exe)


@pytest.mark.parametrize("prec,centre,width,max_iter,waves", CASES)
def test_blocks_match_checked_loop(model, prec, centre, width, max_iter, waves):
    run = subprocess.run([model, str(prec), *centre, width, str(max_iter), str(waves), "5"],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert run.returncode == 0, run.stdout[-2000:]
    fields = dict(zip(run.stdout.split()[::2], map(int, run.stdout.split()[1::2])))
    if centre == CENTRE and width == "1e-6":  # the frames meant to reach them do
        assert fields["cycles"] > 0 and fields["rebases"] > 0
