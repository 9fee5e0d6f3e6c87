"""Registers of the row kernels, from the metadata of the objects built here: a count that costs a wave per SIMD goes unnoticed
in every test of results.  CPU only."""
import os
import re
import subprocess

import pytest

from tritonformer_amd import _build

LLVM = os.path.join(os.path.dirname(os.path.dirname(_build.HIPCC)), "llvm", "bin")


run = lambda *cmd: subprocess.run(cmd, check=True, capture_output=True, text=True).stdout


def code_object(name, d):
    """The device code of csrc/<name>.hip; `d`: a folder for what is unpacked"""
    obj, src = os.path.join(_build.OBJ_DIR, f"{name}.o"), os.path.join(_build.CSRC, f"{name}.hip")
    if not os.path.exists(obj) or os.path.getmtime(obj) < os.path.getmtime(src):
        pytest.skip(f"no object of csrc/{name}.hip as it is: only the linked library is here")
    fat, code = str(d / "fat"), str(d / "code")
    run(f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, str(d / "copy.o"))
    run(f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
        f"--input={fat}", f"--output={code}")
    return code


def kernels_of(name, d):
    """{mangled name: (vector registers, bytes of scratch)} of csrc/<name>.hip"""
    notes = run(f"{LLVM}/llvm-readelf", "--notes", code_object(name, d))
    found = re.findall(r"\.name:\s+(\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)(?:\n\s+\..*)*?\n\s+\.vgpr_count:\s+(\d+)",
                       notes)
    return {name: (int(regs), int(scratch)) for name, scratch, regs in found}


def listings(code):
    """{mangled name: [(address, mnemonic, operands, branch target | None)]}"""
    kernels, current, base = {}, None, 0
    for line in run(f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", code).splitlines():
        head = re.match(r"([0-9a-f]+) <(\S+)>:$", line)
        text, _, note = line.partition("//")
        if head:
            base, current = int(head[1], 16), kernels.setdefault(head[2], [])
        elif note:
            mnemonic, _, operands = text.strip().partition(" ")
            target = re.search(r"\+0x([0-9a-f]+)>$", note) if "branch" in mnemonic else None
            current.append((int(note.split(":")[0], 16), mnemonic, operands, base + int(target[1], 16) if target else None))
    return kernels


def touched_in_flight(listing):
    """Addresses of instructions that touch a register whose LDS read may be in flight, over all paths.  What is tracked per register
    is the least number of LDS operations after its read: these return in order, so a wait that leaves N in flight leaves only
    reads with fewer than N after them.  (Other operations that the counter counts only make a wait longer.)"""
    regs = lambda text: {(k, r) for k, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))(?!\w)", text)
                         for r in (range(int(lo), int(hi) + 1) if lo else (int(one),))}
    steps = []
    for at, mnemonic, operands, _ in listing:
        wait = re.search(r"lgkmcnt\((\d+)\)", operands) if mnemonic == "s_waitcnt" else None
        lds = mnemonic.startswith("ds_")
        reads = regs(operands.split(",")[0]) if lds and not mnemonic.startswith("ds_write") else ()
        steps.append((at, regs(operands), int(wait[1]) if wait else None, lds, reads))
    index = {at: i for i, (at, *_) in enumerate(listing)}
    joins = {index[target] for *_, target in listing if target is not None}
    seen, todo, found = {}, [(0, {})], set()
    while todo:
        i, flying = todo.pop()
        while i < len(steps):
            if i in joins:  # a place that several paths reach: on from there with the worst of all, if that is news
                old = seen.get(i)
                if old is not None:
                    if all(old.get(r, 99) <= age for r, age in flying.items()):
                        break
                    flying = {r: min(flying.get(r, 99), old.get(r, 99)) for r in {**flying, **old}}
                seen[i] = dict(flying)
            at, used, wait, lds, reads = steps[i]
            if flying and any(r in flying for r in used):
                found.add(at)
            if wait is not None:
                flying = {r: age for r, age in flying.items() if age < wait}
            if lds:
                flying = {r: age + 1 for r, age in flying.items()}
                flying.update((r, 0) for r in reads)
            _, mnemonic, _, target = listing[i]
            if target is not None:
                todo.append((index[target], dict(flying)))
            if mnemonic in ("s_endpgm", "s_branch"):
                break
            i += 1
    return found


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


@pytest.fixture(scope="module")
def gemm_code(tmp_path_factory):
    return listings(code_object("gemm", tmp_path_factory.mktemp("gemm")))


def test_gemm_of_wide_and_of_ragged_rows_keeps_two_waves_per_simd(tmp_path):
    kernels = {k: v for k, v in kernels_of("gemm", tmp_path).items() if re.search("gemm_(wide|reg)_", k)}
    assert len(kernels) == 2 * 4 * (1 + 3)
    # register-staged 256x256 with just one operand contraction-strided: seven registers, not in the loop over whole stages
    allowed = lambda k: 32 if re.search(r"Li256ELi256E.*(Lb1ELb0E|Lb0ELb1E)E", k) else 0
    assert {k: v for k, v in kernels.items() if v[0] > 256 or v[1] > allowed(k)} == {}


def test_gemm_touches_no_fragment_in_flight(gemm_code):
    """The kernels request fragments ahead of counted waits, in registers that the compiler takes as written: a spill, a copy or a use
    ahead of its wait would see what was there before."""
    kernels = {k: v for k, v in gemm_code.items() if re.search("gemm_(dma|wide|reg)_", k)}
    assert len(kernels) == 2 * (4 * 6 + 1) + 8 + 24
    assert {k: sorted(map(hex, bad))[:4] for k, v in kernels.items() if (bad := touched_in_flight(v))} == {}


def test_a_fragment_in_flight_is_seen(gemm_code):
    """The check above on a listing with one wait of the main loop taken out of the text."""
    kernel = next(v for k, v in gemm_code.items() if "gemm_dma_kernelIDF16_Li256ELi256E" in k)
    waits = [i for i, (_, m, ops, _) in enumerate(kernel) if m == "s_waitcnt" and re.search(r"lgkmcnt\(([1-9]\d*)\)", ops)]
    assert len(waits) > 8
    assert all(touched_in_flight(kernel[:i] + kernel[i + 1:]) for i in waits[:8])
