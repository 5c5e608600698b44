"""What the compiler puts around the inline assembly of the matrix kernels.

Its hazard recogniser pads wait states between the instructions that it forms itself and looks at none inside inline
assembly.  gfx950 asks for several of them between a matrix instruction and a vector instruction that writes a register
the former still reads or writes, and for two between a vector instruction that writes a scalar register
(v_readlane_b32: a spilled one that comes back) and a vector instruction that reads it.  So inline assembly in a kernel
with matrix instructions holds no vector ALU instruction, and its memory instructions take no address from scalar
registers (five wait states after a vector instruction that wrote them)."""
import re
import subprocess

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


def test_inline_assembly_of_the_matrix_kernels_needs_no_wait_states(tmp_path):
    out = tmp_path / "prefill.s"
    subprocess.run([build._hipcc(), *build.COMMON_FLAGS, "--cuda-device-only", "-S", str(build.CSRC / "prefill.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    assembly = out.read_text()
    kernels, found = _hazards(assembly)
    assert len(kernels) > 20 and "global_load_lds_dwordx4" in assembly   # the scan met what it looks for
    assert not found, f"{len(found)} lines, first {found[:3]}"
