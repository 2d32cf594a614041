"""The FP64 block loops have their 8-byte instructions at multiples of 8 bytes: a wave that
is alone on its SIMD takes 10 to 18 % longer over a block at odd multiples of 4.  Looked up
in the assembly of the built modules."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def straight_runs(path, tmp_path):
    """Per kernel, the stretches of instructions between branches, as (address, mnemonic)."""
    code = str(tmp_path / "code.o")
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--type=o", "--unbundle", f"--input={path}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={code}"], check=True)
    text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", code], check=True,
                          stdout=subprocess.PIPE, text=True).stdout
    kernels, runs = {}, None
    for line in text.splitlines():
        head = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if head:
            runs = kernels.setdefault(head.group(1), [[]])
            continue
        found = re.match(r"\s+(\S+).*// ([0-9A-F]+):", line)
        if not found or runs is None:
            continue
        if found.group(1).startswith(("s_branch", "s_cbranch", "s_endpgm")):
            runs.append([])
        else:
            runs[-1].append((int(found.group(2), 16), found.group(1)))
    return kernels


@pytest.mark.parametrize("module,kernels,block", [
    ("escape_family", r"escapeTilesPersistentDouble\w+K8", 8), ("escape_family", r"escapeTilesPersistentDouble\w+K16", 16),
    ("escape_family", r"escapeTilesPersistentDouble\w+K32", 32), ("escape_family", r"escapeDrainDouble\w+K8", 8),
    ("escape_family", r"escapeDrainDouble\w+K16", 16), ("escape_family", r"escapeTile(Samples)?Double[A-Z][a-z]+", 16),
    ("escape_family", r"escapeTileSamplesDouble\w+K8", 8), ("escape_family", r"escapePass[1Q]Double\w+K16", 16),
    ("escape_family", r"escapePass[1Q]Double\w+K8", 8), ("escape_family", r"deepDirectDouble\w+", 16), ("mandelbrot", r"fractalRender\w+Double\w*", 16),
    ("julia", r"fractalRender\w+Double\w*", 16)])
def test_blocks_start_at_multiples_of_eight(tmp_path, module, kernels, block):
    path = os.path.join(ROOT, "chaos-ultra_amd", "kernels", module + ".hsaco")
    seen = 0
    for name, runs in straight_runs(path, tmp_path).items():
        if not re.fullmatch(kernels, name):
            continue
        for run in runs:
            steps = [at for at, op in run if op.endswith("_f64") or "_f64_e" in op]
            # six operations a step fused, seven exact, and at most three that test the end
            if any(0 <= len(steps) - k * block <= 3 for k in (6, 7)):
                seen += 1
                assert sum(at % 8 != 0 for at in steps) <= 1, (name, hex(steps[0]))
    assert seen >= 2, "no block found: has the step's operation count changed?"
