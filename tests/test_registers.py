"""What the kernels whose rows live in registers were compiled to: spilled registers are trips to memory."""
import re
import subprocess

import pytest

from kascade_amd import build


@pytest.fixture(scope="module")
def selection(tmp_path_factory):
    """(name, bytes of scratch) of every kernel of topk.hip"""
    out = tmp_path_factory.mktemp("asm") / "topk.s"
    subprocess.run([build._hipcc(), *build.COMMON_FLAGS, "--cuda-device-only", "-S", str(build.CSRC / "topk.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    return re.findall(r"\.name: +(_Z\S+)\n.*?\.private_segment_fixed_size: (\d+)", out.read_text(), re.S)


@pytest.mark.parametrize("kernel,instances", [("topk_select_reg_kernel", 9), ("decode_pool_select_kernel", 5), ("topk_split_", 7)])
def test_selection_keeps_its_row_in_registers(selection, kernel, instances):
    """None of them uses scratch, up to 16 chunks of 8 entries a thread; nor do the passes over long rows' chunks."""
    found = [(name, scratch) for name, scratch in selection if kernel in name]
    assert len(found) == instances
    assert all(scratch == "0" for _, scratch in found), found
