"""Registers of the row kernels, from the metadata of the objects built here: a count that costs a wave per SIMD goes unnoticed
in every test of results.  CPU only."""
import os
import re
import subprocess

import pytest

from tritonformer_amd import _build

LLVM = os.path.join(os.path.dirname(os.path.dirname(_build.HIPCC)), "llvm", "bin")


@pytest.fixture(scope="module")
def norm_kernels(tmp_path_factory):
    """{mangled name: (vector registers, bytes of scratch)} of csrc/norm.hip"""
    obj, src = os.path.join(_build.OBJ_DIR, "norm.o"), os.path.join(_build.CSRC, "norm.hip")
    if not os.path.exists(obj) or os.path.getmtime(obj) < os.path.getmtime(src):
        pytest.skip("no object of csrc/norm.hip as it is: only the linked library is here")
    d = tmp_path_factory.mktemp("norm")
    fat, code = str(d / "norm.fat"), str(d / "norm.co")
    run = lambda *cmd: subprocess.run(cmd, check=True, capture_output=True, text=True).stdout
    run(f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, str(d / "copy.o"))
    run(f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
        f"--input={fat}", f"--output={code}")
    notes = run(f"{LLVM}/llvm-readelf", "--notes", code)
    found = re.findall(r"\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)(?:\n\s+\..*)*?\n\s+\.vgpr_count:\s+(\d+)",
                       notes)
    return {name: (int(regs), int(scratch)) for name, scratch, regs in found}


def test_layernorm_backward_keeps_two_waves_per_simd(norm_kernels):
    """A SIMD holds 512 registers per lane: beyond 256 the workgroup of four waves has the CU to itself."""
    kernels = {k: v for k, v in norm_kernels.items() if "ln_bwd_vec" in k}
    assert len(kernels) == 80  # 4 pairs of types, 5 row widths, with and without a residual, whole and ragged rows
    assert {k: v for k, v in kernels.items() if v[0] > 256 or v[1]} == {}


def test_layernorm_forward_of_ragged_rows_and_fp32_parameters_keeps_four_waves_per_simd(norm_kernels):
    kernels = {k: v for k, v in norm_kernels.items() if re.search(r"ln_fwd_vecIDF16b?_?fLi\dELi\dELb\dELb1E", k)}
    assert len(kernels) == 20
    assert {k: v for k, v in kernels.items() if v[0] > 128 or v[1]} == {}
