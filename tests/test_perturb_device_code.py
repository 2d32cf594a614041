"""The perturbation kernels' own code, compiled for the CPU and run on 64-lane waves in
lockstep (tests/emulate/perturb_simt.cpp), against the oracle.

The reference orbit's entries, the cycle found in it and the blocks' bounds equal the
oracle's orbit and plain restatements; pixels' counts, states and |z|^2 equal the checked
loop's bit for bit, with all of the schedule's shortcuts, without the reference's cycle and without
the blocks that leave their tests out; and the views meant to take a shortcut do take it:
without it the waves need more operations across lanes.  Reads past the last entry, and
operations across lanes that not all of them come to, stop the program.
"""
import os
import subprocess

import pytest

from conftest import ROOT

CENTRE = ("-0.743643887037151", "0.131825904205330")
CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")


@pytest.fixture(scope="module")
def waves(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("simt") / "perturb_simt")
    emulate, oracle = os.path.join(ROOT, "tests", "emulate"), os.path.join(ROOT, "oracle")
    build = subprocess.run([CLANG, "-std=c++17", "-O2", "-ffp-contract=off", "-mfma", "-Wall", "-Wextra",
                            "-Wno-unused-function", f"-I{os.path.join(emulate, 'simt')}",
                            os.path.join(emulate, "perturb_simt.cpp"), "-o", exe, f"-L{oracle}", "-loracle",
                            f"-Wl,-rpath,{oracle}"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if build.returncode != 0:
        pytest.fail(build.stdout[-4000:])

    def run(precision, centre, width, max_iter, limit=None, n=6, seed=5):
        out = subprocess.run([exe, str(precision), *map(str, centre), str(width), str(max_iter),
                              str(limit or max_iter), str(n), str(seed)], stdout=subprocess.PIPE,
                             stderr=subprocess.STDOUT, text=True, timeout=120)
        assert out.returncode == 0, out.stdout
        words = out.stdout.split()
        return dict(zip(words[::2], map(int, words[1::2])))

    return run


# references that settle into cycles: their period, and how far from the start at most; the
# second limit is a frame that keeps a longer orbit
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("limit", [9001, 2999])
@pytest.mark.parametrize("centre,width,period,start", [
    ((-0.4, 0.05), 0.9, 1, 100), ((-1.02, 0.03), 0.3, 2, 100), ((-0.123, 0.745), 0.12, 3, 100),
    ((0.2823, 0.5301), 0.05, 4, 100), ((-0.5355, 0.6085), 0.02, 10, 1000),
    ((-0.7436440753, 0.1318253789), 1e-6, 78, 2000)])
def test_along_a_periodic_reference(waves, precision, centre, width, period, start, limit):
    r = waves(precision, centre, width, 9001, limit)
    assert r["first_period"] == period and r["from"] <= start
    if period <= 4:  # the pixels' orbits come back within the limit
        assert 2 * r["operations"] < r["uncycled"]


# frames whose deltas stay far below the reference's values for many blocks
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("centre,width,max_iter", [
    (CENTRE, 1e-12, 4001), (CENTRE, 1e-25, 1000), (CENTRE, 1e-10, 5000), ((0.2501, 0.0), 1e-5, 999)])
def test_blocks_without_tests(waves, precision, centre, width, max_iter):
    r = waves(precision, centre, width, max_iter)
    assert r["bounded"] > 0 and r["operations"] < r["tested"]


def test_the_bounds_matter(waves):
    """With no test run at all, pixels do come out wrong."""
    assert waves(64, CENTRE, 1e-12, 4001)["unsound"] > 0


# frequent rebases, interior pixels with a reference that escapes, references of a few steps,
# limits around a block's length and around the reference's own
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("centre,width,max_iter,n", [
    (CENTRE, 1e-6, 30000, 3), (CENTRE, 1.0, 2000, 12), ((-0.25, 0.125), 1.0, 2000, 12), ((0.5, 0.0), 1e-3, 2000, 6),
    ((0.7, 0.3), 0.01, 2000, 6), ((0.3, 0.02), 0.3, 3000, 12), ((0.26, 0.001), 0.05, 4000, 8),
    ((-1.0, 0.0), 0.5, 700, 12), ((0.0, 0.0), 0.5, 97, 6), ((0.0, 1.0), 1e-10, 700, 4), ((1.2, 0.5), 1.0, 100, 8),
    *[((0.5, 0.5), 0.5, k, 6) for k in (1, 2, 7, 8, 9, 10, 31, 32, 33)],
    *[((0.3, 0.02), 0.3, k, 6) for k in (28, 29, 30, 31, 32, 33, 61, 62, 63, 64, 65)],
    *[(CENTRE, 1e-3, k, 6) for k in (1, 31, 32, 33, 63, 64, 65)]])
def test_frames(waves, precision, centre, width, max_iter, n):
    waves(precision, centre, width, max_iter, n=n)


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("centre,width", [((0.5, 0.5), 0.05), ((-1.2, 0.6), 0.1), ((0.9, 0.9), 0.5), ((0.7, 0.3), 0.01)])
def test_frames_beside_the_set_take_no_blocks(waves, precision, centre, width):
    """A reference of a few steps, and pixels that escape with it: one operation a checked
    step and a few besides, where a block of 32 and its replay take 46."""
    r = waves(precision, centre, width, 200, n=8)
    assert r["last"] <= 7 and r["operations"] <= 8 * (r["last"] + 10)
