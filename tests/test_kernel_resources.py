"""Registers decide how many wavefronts a SIMD holds: the general field-array
kernels (non-uniform axes, several terms), the EHSS kernels and the batch kernel
with mixtures and arrays keep theirs."""
import os
import re
import shutil
import subprocess

import pytest

from icarion_amd import build

OBJ = os.path.join(build.OBJDIR, "step_kernels.o")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLER = "/opt/rocm/llvm/bin/clang-offload-bundler"


@pytest.fixture(scope="module")
def vgprs(tmp_path_factory):
    if not (os.path.exists(OBJ) and os.path.exists(READELF) and os.path.exists(BUNDLER) and shutil.which("c++filt")):
        pytest.skip("no object of this build or no LLVM tools")
    co = str(tmp_path_factory.mktemp("co") / "step.co")
    fat = co + ".fatbin"
    subprocess.run(["objcopy", "-O", "binary", "--only-section=.hip_fatbin", OBJ, fat], check=True)
    subprocess.run([BUNDLER, "--unbundle", "--type=o", f"--input={fat}", f"--output={co}",
                    f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}"], check=True)
    notes = subprocess.run([READELF, "--notes", co], check=True, capture_output=True, text=True).stdout
    out = {}
    for block in notes.split("- .agpr_count:")[1:]:
        name = re.search(r"\.name:\s+(\S+)", block).group(1)
        out[name] = int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1))
    names = subprocess.run(["c++filt"] + list(out), check=True, capture_output=True, text=True).stdout.splitlines()
    return {re.sub(r"^void icarion::|\(.*", "", n): v for n, v in zip(names, out.values())}


# 512 registers per SIMD lane, given out in eights
@pytest.mark.parametrize("kernel,waves", [
    ("step_f32_kernel<0, 3, 0, false>", 3), ("step_f32_kernel<0, 3, 1, false>", 3), ("step_f32_kernel<0, 3, 3, false>", 3),
    ("step_f32_kernel<1, 3, 0, false>", 3), ("step_f32_kernel<1, 3, 1, false>", 3), ("step_f32_kernel<1, 3, 3, false>", 3),
    ("step_f64_kernel<1, 3, 1, false>", 2), ("step_f64_kernel<1, 3, 4, false>", 2), ("step_f64_kernel<0, 0, 5, false>", 2),
    ("step_f64_kernel<0, 0, 6, false>", 2), ("batch_kernel<1, true>", 3),
    ("step_f64_ehss_kernel<0, 0>", 2), ("step_f64_ehss_kernel<1, 2>", 2)])
def test_wavefronts_per_simd(vgprs, kernel, waves):
    assert 512 // (-(-vgprs[kernel] // 8) * 8) >= waves, vgprs[kernel]
