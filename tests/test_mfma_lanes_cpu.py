"""The NNP force kernels' 4x4x1 matrix products take their coefficient rows
from all four lanes of a block, and an MFMA reads every lane's registers
whatever the exec mask: the products have to run with no lane masked off, or
rows come from registers that the compiler does not keep.  Checked in the
assembly of the library as built here."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "cabanamd_amd", "libcabanamd_amd.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"

# an exec mask is narrowed by these and widened by s_or / s_mov
NARROWS = re.compile(r"\b(s_\w*saveexec_b64|s_and(n2)?_b64 exec|s_xor_b64 exec)\b")
EXEC = re.compile(r"\b(s_\w*saveexec_b64|s_\w+_b64 exec)\b")


def _listing(tmp):
    lib = os.path.join(tmp, "lib.so")
    shutil.copy(LIB, lib)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp, check=True,
                   stdout=subprocess.DEVNULL)
    for f in sorted(os.listdir(tmp)):
        if "gfx950" in f:
            yield from subprocess.run(
                [OBJDUMP, "-d", "--mcpu=gfx950", os.path.join(tmp, f)], check=True,
                stdout=subprocess.PIPE, text=True).stdout.splitlines()


def test_force_products_run_in_all_lanes(tmp_path):
    if not os.path.exists(OBJDUMP) or not os.path.exists(LIB):
        pytest.skip("needs llvm-objdump and the built library")
    kernel, narrowed, seen = None, False, {}
    for line in _listing(str(tmp_path)):
        m = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        if m:
            kernel, narrowed = m.group(1), False
        elif EXEC.search(line):
            narrowed = bool(NARROWS.search(line))
        elif "v_mfma_f32_4x4x1" in line:
            seen.setdefault(kernel, []).append(narrowed)
    # one to eight etas, one and four waves on an atom
    assert len(seen) == 16, sorted(seen)
    for kernel, masked in seen.items():
        assert "k_nnp_force_pow" in kernel
        assert not any(masked), f"{kernel}: {sum(masked)} of {len(masked)} under a mask"
