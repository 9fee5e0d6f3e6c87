"""Registers of the row kernels, from the metadata of the objects built here: a count that costs a wave per SIMD goes unnoticed
in every test of results.  CPU only."""
import os
import re
import subprocess

import pytest

from tritonformer_amd import _build

LLVM = os.path.join(os.path.dirname(os.path.dirname(_build.HIPCC)), "llvm", "bin")


def kernels_of(name, d):
    """{mangled name: (vector registers, bytes of scratch)} of csrc/<name>.hip; `d`: a folder for what is unpacked"""
    obj, src = os.path.join(_build.OBJ_DIR, f"{name}.o"), os.path.join(_build.CSRC, f"{name}.hip")
    if not os.path.exists(obj) or os.path.getmtime(obj) < os.path.getmtime(src):
        pytest.skip(f"no object of csrc/{name}.hip as it is: only the linked library is here")
    fat, code = str(d / "fat"), str(d / "code")
    run = lambda *cmd: subprocess.run(cmd, check=True, capture_output=True, text=True).stdout
    run(f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, str(d / "copy.o"))
    run(f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
        f"--input={fat}", f"--output={code}")
    notes = run(f"{LLVM}/llvm-readelf", "--notes", code)
    found = re.findall(r"\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)(?:\n\s+\..*)*?\n\s+\.vgpr_count:\s+(\d+)",
                       notes)
    return {name: (int(regs), int(scratch)) for name, scratch, regs in found}


@pytest.fixture(scope="module")
def norm_kernels(tmp_path_factory):
    return kernels_of("norm", tmp_path_factory.mktemp("norm"))


def test_layernorm_backward_keeps_two_waves_per_simd(norm_kernels):
    """A SIMD holds 512 registers per lane: beyond 256 the workgroup of four waves has the CU to itself."""
    kernels = {k: v for k, v in norm_kernels.items() if "ln_bwd_vec" in k}
    assert len(kernels) == 80  # 4 pairs of types, 5 row widths, with and without a residual, whole and ragged rows
    assert {k: v for k, v in kernels.items() if v[0] > 256 or v[1]} == {}


def test_layernorm_forward_of_ragged_rows_and_fp32_parameters_keeps_four_waves_per_simd(norm_kernels):
    kernels = {k: v for k, v in norm_kernels.items() if re.search(r"ln_fwd_vecIDF16b?_?fLi\dELi\dELb\dELb1E", k)}
    assert len(kernels) == 20
    assert {k: v for k, v in kernels.items() if v[0] > 128 or v[1]} == {}


def test_cross_entropy_forward_of_whole_rows_holds_a_row_and_little_else(tmp_path):
    """Five registers per chunk of the row, eight more: what the compiler needs where it follows one test per chunk."""
    kernels = {k: v for k, v in kernels_of("ce", tmp_path).items() if re.search(r"ce_fwd_regsIDF16b?_?Li\d+ELb0ELb0E", k)}
    assert len(kernels) == 6
    assert {k: v for k, v in kernels.items() if v[0] > 5 * int(re.search(r"Li(\d+)E", k)[1]) + 8 or v[1]} == {}


def test_direct_to_lds_gemm_keeps_two_waves_per_simd_and_spills_nothing(tmp_path):
    """Fragments are in flight in registers that the compiler takes as written: a spill or a copy of one would read it too early."""
    kernels = {k: v for k, v in kernels_of("gemm", tmp_path).items() if "gemm_dma_" in k}
    assert len(kernels) == 2 * (4 * 6 + 1)  # two types; four operand layouts of six tiles, the grouped launch
    assert {k: v for k, v in kernels.items() if v[0] > 256 or v[1]} == {}
