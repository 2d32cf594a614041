"""The host's rules for the form of a launch, at frames measured with each form: a launch
must not take the slower one where that cost more than a few per cent."""
import os
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "launch_rules")
    build = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__",
                            f"-I{ROCM}/include", os.path.join(ROOT, "tests", "emulate", "launch_rules.cpp"),
                            "-o", exe, f"-L{ROCM}/lib", "-lamdhip64", f"-Wl,-rpath,{ROCM}/lib"],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if build.returncode != 0:
        pytest.fail(build.stdout[-4000:])
    return lambda *args: int(subprocess.run([exe, *map(str, args)], check=True, stdout=subprocess.PIPE,
                                            text=True).stdout)


@pytest.mark.parametrize("size,samples,max_iter,reuse,overlap,groups", [
    # zoom frames: deep ones wait for the fovea, shallow ones pay for twice the waves
    ((1920, 1080), 4, 5000, 1, 0.95, 1), ((1280, 720), 4, 5000, 1, 0.95, 1), ((320, 240), 4, 300, 1, 0.95, 1),
    ((3840, 2160), 4, 1600, 1, 0.95, 2), ((2560, 1440), 5, 900, 1, 0.95, 2), ((1920, 1080), 5, 900, 1, 0.95, 2),
    ((1280, 720), 4, 900, 1, 0.95, 2), ((640, 360), 1, 5000, 1, 0.95, 2),
    # little of the earlier frame is left: as whole frames
    ((1920, 1080), 4, 5000, 1, 0.3, 2), ((640, 360), 4, 5000, 1, 0.3, 1),
    # whole frames
    ((1280, 720), 4, 5000, 0, 0, 1), ((800, 480), 4, 5000, 0, 0, 1), ((1024, 576), 5, 1600, 0, 0, 1),
    ((640, 360), 5, 900, 0, 0, 1), ((160, 120), 8, 300, 0, 0, 1), ((800, 480), 5, 900, 0, 0, 2),
    ((1024, 576), 8, 900, 0, 0, 2), ((640, 360), 8, 300, 0, 0, 2), ((1920, 1080), 4, 50000, 0, 0, 2),
    ((800, 480), 1, 5000, 0, 0, 2)])
def test_render_forms(rule, size, samples, max_iter, reuse, overlap, groups):
    assert rule("forms", *size, samples, max_iter, reuse, overlap) == groups


@pytest.mark.parametrize("blocks,per_cu,bytes_", [
    (1, 4, 0), (4 * 256, 4, 0), (10 * 256 - 1, 4, 0), (10 * 256, 4, 40960), (28 * 256, 4, 40960),
    (28 * 256 + 1, 4, 0), (10 * 256, 6, 26880), (1 << 40, 4, 0)])
def test_unused_lds(rule, blocks, per_cu, bytes_):
    """Asked for only by launches of 10 to 28 blocks per CU: it keeps other streams' kernels off
    the CUs, and smaller launches have nothing to hold back."""
    assert rule("lds", blocks, 10, 28, per_cu) == bytes_
