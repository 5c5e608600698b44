"""What the compiler puts around the inline assembly of the matrix kernels.

Its hazard recogniser pads wait states between the instructions that it forms itself and looks at none inside inline
assembly.  gfx950 asks for several of them between a matrix instruction and a vector instruction that writes a register
the former still reads or writes, and for two between a vector instruction that writes a scalar register
(v_readlane_b32: a spilled one that comes back) and a vector instruction that reads it.  So inline assembly in a kernel
with matrix instructions holds no vector ALU instruction, and its memory instructions take no address from scalar
registers (five wait states after a vector instruction that wrote them)."""
import re
import subprocess

import pytest

from kascade_amd import build

SGPR = re.compile(r"\bs(\d+\b|\[\d+:\d+\])")


def _hazards(assembly):
    """(kernels with matrix instructions, lines of inline assembly in them that no wait state protects)"""
    kernels, found, kernel, inline, lines = set(), [], None, False, []
    for line in assembly.splitlines():
        text = line.split(";", 1)[0].strip()
        if line.startswith("_Z") and text.endswith(":"):
            kernel, lines = text[:-1], []
        elif "#ASMSTART" in line or "#ASMEND" in line:
            inline = "#ASMSTART" in line
        elif line.startswith(".Lfunc_end"):
            found += lines if kernel in kernels else []
        elif text.startswith("v_mfma"):
            kernels.add(kernel)
        elif inline and (text.startswith("v_") or (re.match(r"(global|buffer|flat|scratch)_", text) and SGPR.search(text))):
            lines.append(f"{kernel}: {text}")
    return kernels, found


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "prefill.s"
    subprocess.run([build._hipcc(), *build.COMMON_FLAGS, "--cuda-device-only", "-S", str(build.CSRC / "prefill.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    return out.read_text()


def test_inline_assembly_of_the_matrix_kernels_needs_no_wait_states(assembly):
    kernels, found = _hazards(assembly)
    assert len(kernels) > 20 and "global_load_lds_dwordx4" in assembly   # the scan met what it looks for
    assert not found, f"{len(found)} lines, first {found[:3]}"


def test_log_sum_units_of_32_queries_fit_four_to_a_compute_unit(assembly):
    """The order of the units counts on four workgroups of the pass for log-sums alone per compute unit: 128
    vector registers, none of them spilled, strided and paged, at both head dims, in both types, with and without head
    slots that no query head fills."""
    kernels = re.findall(r"\.name: +(\S+prefill_attn_kernel_q32ILb0ELb0E\S+)\n.*?\.private_segment_fixed_size: (\d+)"
                         r".*?\.vgpr_count: +(\d+)", assembly, re.S)
    assert len(kernels) == 16
    assert all(int(vgprs) <= 128 and scratch == "0" for _, scratch, vgprs in kernels), kernels


def test_whole_groups_run_no_kernel_for_spare_head_slots(assembly):
    """Every attention kernel is there with and without head slots that no query head fills: the second loop of the
    former costs groups that fill whole four slots its registers, in passes that report log-sums too."""
    found = re.findall(r"\.name: +\S+prefill_attn_kernel_q(32ILb\dELb\dE|64I)Lb(\d)ELi(\d+)E(DF16_|DF16b)Lb(\d)E(Lb\dE)?E", assembly)
    whole, spare = ({(a, b, c, d, f) for a, b, c, d, s, f in found if s == slot} for slot in "01")
    assert whole == spare and len(whole) == 36
