"""How many wavefronts of a kernel a compute unit holds, by the registers and the LDS the compiler's notes in the built library give: where the
figures beside the kernels rest on it, a change that takes a place away is to be seen."""
import os
import re
import shutil
import subprocess

import pytest

from svox_amd.csrc import _abi

LLVM = "/opt/rocm/llvm/bin"
SIMDS, REGISTERS, LDS, GRANULE = 4, 512, 160 * 1024, 1280


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """demangled name -> (bytes of LDS, registers, threads of a block)"""
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no LLVM tools")
    at = str(tmp_path_factory.mktemp("library"))
    shutil.copy(_abi.LIB_PATH, at)
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", os.path.basename(_abi.LIB_PATH)], cwd=at, check=True, capture_output=True)
    found = {}
    for f in sorted(os.listdir(at)):
        if f.endswith("gfx950"):
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", os.path.join(at, f)], check=True, capture_output=True, text=True).stdout
            for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
                number = lambda key: int(re.search(rf"\.{key}:\s+(\d+)", kernel).group(1))
                found[re.search(r"\.symbol:\s+'?(\S+?)\.kd", kernel).group(1)] = (number("group_segment_fixed_size"), number("vgpr_count"),
                                                                                 number("max_flat_workgroup_size"))
    names = subprocess.run(["c++filt"], input="\n".join(found), check=True, capture_output=True, text=True).stdout.split("\n")
    return {re.sub(r"^void |svox::|\(.*", "", name): found[symbol] for name, symbol in zip(names, found)}


def wavefronts(kernel):
    lds, registers, threads = kernel
    waves = threads // 64
    by_registers = SIMDS * min(8, REGISTERS // (-(-registers // 8) * 8))
    by_lds = LDS // (-(-lds // GRANULE) * GRANULE) * waves if lds else 32
    return min(by_registers // waves * waves, by_lds)


# (the rays in pieces of double precision: group_kernels.h)
@pytest.mark.parametrize("basis,forward,backward", [(0, 9, 9), (1, 9, 9), (4, 9, 9), (9, 8, 8), (16, 8, 8), (25, 8, 7)])
@pytest.mark.parametrize("source", ["BatchSource<double>", "ImageSource<double>"])
def test_double_precision_rays_in_pieces(kernels, basis, forward, backward, source):
    assert wavefronts(kernels[f"render_group_kernel<{basis}, {source}, false>"]) >= forward
    assert wavefronts(kernels[f"render_group_kernel<{basis}, {source}, true>"]) >= backward
