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


def by_lds(kernel):
    return LDS // (-(-kernel[0] // GRANULE) * GRANULE) * (kernel[2] // 64)


# (a path of 11 levels and its dump rows, beside the shading's lists: MarchShared, SplitBox)
@pytest.mark.parametrize("policy,walks_and_shades,splits,marches", [("0, 0", 18, 24, 21), ("1, 1", 18, 24, 21), ("1, 4", 18, 24, 18), ("1, 9", 18, 24, 16), ("1, 16", 18, 24, 14),
                                                                    ("1, 25", 18, 24, 11), ("2, 1", 21, 24, 21), ("2, 4", 18, 22, 18), ("2, 9", 16, 20, 16),
                                                                    ("2, 16", 14, 16, 14), ("2, 25", 11, 16, 11)])
@pytest.mark.parametrize("source", ["BatchSource<float>", "ImageSource<float>"])
def test_wavefronts_lds_has_room_for(kernels, policy, walks_and_shades, splits, marches, source):
    policy = f"OctreePolicy<{policy}>"
    for refill in ("false", "true"):
        for noted in ("false", "true"):
            assert by_lds(kernels[f"render_forward_kernel<{policy}, {source}, false, {refill}, {noted}, false, false>"]) >= walks_and_shades
            assert by_lds(kernels[f"render_forward_split_kernel<{policy}, {source}, {noted}, false>"]) >= splits
        for mode in (0, 1):
            assert by_lds(kernels[f"render_backward_kernel<{policy}, {source}, {refill}, {mode}>"]) >= marches
        assert by_lds(kernels[f"se_grad_kernel<{policy}, {source}, {refill}>"]) >= marches


@pytest.mark.parametrize("policy,notes,marches", [("0, 0", 16, 20), ("1, 16", 16, 14), ("2, 4", 16, 16), ("2, 9", 16, 16), ("2, 16", 14, 14)])
@pytest.mark.parametrize("source", ["BatchSource<float>", "ImageSource<float>"])
def test_wavefronts_that_take_notes_or_march_without(kernels, policy, notes, marches, source):
    for refill in ("false", "true"):
        for mode in (0, 1):
            assert wavefronts(kernels[f"render_backward_kernel<OctreePolicy<{policy}>, {source}, {refill}, {mode}>"]) >= marches
        if policy.startswith("2"):
            for grad in ("false", "true"):
                assert wavefronts(kernels[f"render_forward_kernel<OctreePolicy<{policy}>, {source}, false, {refill}, true, {grad}, false>"]) >= notes


@pytest.mark.parametrize("policy,walks,takes_new_rays", [("0, 0", 20, 16), ("1, 1", 20, 16), ("1, 4", 18, 16), ("2, 1", 20, 16), ("2, 4", 18, 16), ("2, 9", 16, 16)])
@pytest.mark.parametrize("source", ["BatchSource<float>", "ImageSource<float>"])
def test_wavefronts_of_squared_errors_without_notes(kernels, policy, walks, takes_new_rays, source):
    for refill, most in (("false", walks), ("true", takes_new_rays)):
        assert wavefronts(kernels[f"se_grad_kernel<OctreePolicy<{policy}>, {source}, {refill}>"]) >= most


# (render_forward_kernel: four to a SIMD, as many as a batch of 1 Mi rays has, and not a fifth)
def test_wavefronts_that_take_new_rays_are_four_to_a_simd(kernels):
    kernel = kernels["render_forward_kernel<OctreePolicy<1, 16>, BatchSource<float>, false, true, false, false, false>"]
    assert SIMDS * (REGISTERS // (-(-kernel[1] // 8) * 8)) == 16
