"""KernelArgs reads a kernel's arguments at the address that only a kernel has:
in a function that is called instead of inlined it would be null. Compiled with
the optimiser's own inlining switched off (as a debug build leaves it out), the
address is still taken in kernels alone.
"""
import re
import subprocess

import pytest

from g4hepem_amd import build


@pytest.mark.parametrize("source", ["hepem_capi.hip", "hepem_shower.hip"])
def test_arguments_are_read_in_kernels_only(source, tmp_path):
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-O3", "-shared")]
    ir = tmp_path / "device.ll"
    subprocess.run([build._hipcc(), *flags, "-O1", "-fno-inline", "--cuda-device-only", "-S", "-emit-llvm", f"-I{build.ROOT / 'include'}",
                    f"-I{build.CSRC}", "-o", str(ir), str(build.CSRC / source)], check=True, stderr=subprocess.DEVNULL)
    taken = {}
    function = ""
    for line in ir.open():
        if line.startswith("define"):
            function = line
        elif "call" in line and "kernarg.segment.ptr" in line:
            taken[re.search(r"@([^\s(]+)\(", function).group(1)] = "amdgpu_kernel" in function
    assert taken
    assert not [name for name, kernel in taken.items() if not kernel]
