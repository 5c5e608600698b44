"""CPU-only checks of the C ABI: the library loads, exports every symbol the header declares,
and rejects bad arguments before touching a GPU (return code -1 + message)."""
import ctypes as C
import math
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "kascade_hip.h")


@pytest.fixture(scope="module")
def lib():
    from kascade_amd import _lib
    if not _lib.LIB_PATH.exists():
        from kascade_amd import build
        build.build()
    return _lib.load()


def _declared_functions():
    import glob
    names = set()
    for path in glob.glob(os.path.join(ROOT, "include", "*.h")):
        text = re.sub(r"/\*.*?\*/", "", open(path).read(), flags=re.S)
        names |= set(re.findall(r"\b(kascade_[a-z0-9_]+)\s*\(", text))
    return sorted(names)


def test_header_symbols_are_exported_and_bound(lib):
    from kascade_amd import _lib
    names = _declared_functions()
    assert len(names) >= 14
    for n in names:
        assert hasattr(lib, n), f"{n} declared under include/ but not exported"
        assert n in _lib.SIGNATURES, f"{n} has no ctypes signature"
    assert sorted(_lib.SIGNATURES) == names


def test_abi_version_and_error_buffer(lib):
    assert lib.kascade_abi_version() >= 1
    assert isinstance(lib.kascade_get_last_error(), bytes)


def test_topk_workspace_sizing(lib):
    assert lib.kascade_topk_workspace_bytes(128, 1000) == 0          # short rows: one workgroup per row
    assert lib.kascade_topk_workspace_bytes(8192, 32768) == 0        # too many rows for the workspace
    n = lib.kascade_topk_workspace_bytes(32, 524288)
    assert n == 4 * 32 * (2048 + 2 + 8 + 16 * 36)   # 16 chunks of 32768 entries


def test_one_launch_selection_ends_where_two_are_faster(lib):
    """The pooling workgroup of a decode anchor takes a row's tokens for four query heads at a time: groups
    that fill whole fours of one go further than wide or partly filled ones, at few rows."""
    row = lib.kascade_pool_select_row
    assert row(4, 8) == 24576
    assert all(row(g, 8) == 18432 for g in (1, 2, 5, 7, 8, 12, 16))
    assert all(row(g, 64) == 24576 for g in range(1, 17))
    header = re.search(r"#define KASCADE_POOL_SELECT_ROW (\d+)", open(HEADER).read())
    assert all(row(g, r) <= int(header.group(1)) for g in range(1, 17) for r in (1, 8, 1024))


def test_split_rules_have_one_home(lib):
    """The split counts of the Python wrappers and of the host extension come from the library; the two
    numbers that Python holds itself are the header's."""
    from kascade_amd import kernels, strategy
    constants = dict(re.findall(r"#define (KASCADE_[A-Z_]+) (\d+)", open(HEADER).read()))
    assert kernels.GATHER_ROWS_PER_SPLIT == int(constants["KASCADE_GATHER_ROWS_PER_SPLIT"])
    assert strategy.FUSED_MERGE_MAX_SPLITS == int(constants["KASCADE_FUSED_MERGE_MAX_SPLITS"])
    source = open(os.path.join(ROOT, "kascade_amd", "csrc", "native.cpp")).read()
    assert not re.search(r"\b(1664|384|nearbyint)\b", source)
    # the rule in Python; gathers (cap > 0) among the small launches, up to 64 splits and more, and one whose cap asks for more
    for total, longest, cus, per_cu, least, cap in ((128 * 6656, 6656, 256, 2, 512, 0), (8 * 1664, 1664, 256, 2, 512, 1664),
                                                    (8 * 100, 100, 256, 2, 512, 0), (128 * 13184, 13184, 256, 2, 512, 1664),
                                                    (3, 1, 256, 1, 1, 0), (8 * 524288, 524288, 256, 1, 64, 0), (0, 0, 256, 2, 0, 0),
                                                    (8 * 3328, 3328, 256, 2, 512, 1664), (8 * 3328, 3328, 256, 2, 512, 0),
                                                    (8 * 6144, 6144, 256, 2, 512, 1664), (2 * 12032, 12032, 256, 2, 512, 1664),
                                                    (200000, 200000, 256, 2, 512, 1664)):
        per = max(least, total / (per_cu * cus))
        per = min(per, cap) if cap else per
        small = bool(per) and total / per < cus
        if small:
            per = max(min(128, least), total / cus)
        want = max(1, min(256, round(longest / per))) if per else 1
        if small and cap:
            want = min(want, max(64, math.ceil(longest / cap)))
        assert lib.kascade_decode_num_split(total, longest, cus, per_cu, least, cap) == want


def test_known_equal_lists_share_the_rule(lib):
    """Lists known to fill the launch: gathers of up to 6144 rows within 16 splits, few streamed lists one workgroup per unit."""
    for lists, rows, cap, plain, equal in ((8, 3328, 1664, 26, 16), (8, 6144, 1664, 32, 16), (8, 6272, 1664, 32, 32), (8, 1664, 1664, 13, 13),
                                           (8, 65536, 0, 64, 32), (64, 3064, 0, 6, 4), (128, 13184, 1664, 8, 8)):
        assert lib.kascade_decode_num_split(lists * rows, rows, 256, 2, 512, cap) == plain
        assert lib.kascade_decode_num_split_equal(lists, rows, 256, 2, 512, cap) == equal


@pytest.mark.parametrize("lists,rows,splits,cap,want", [
    (64, 3064, 6, 0, 4), (72, 2564, 5, 0, 7), (42, 1664, 8, 1664, 6),            # one round, two, a gather's one
    (64, 3064, 4, 0, 4), (64, 3064, 8, 0, 8), (58, 3064, 8, 0, 8),                # whole rounds, and 464 of 512: as they are
    (208, 5000, 2, 0, 1), (208, 4000, 2, 1664, 2), (208, 1600, 2, 1664, 1),       # one round only where a gather's splits allow it
    (136, 6656, 3, 1664, 3), (176, 6656, 2, 1664, 4), (200, 6656, 2, 1664, 2),    # two rounds or three then
    (264, 896, 1, 1664, 1), (300, 9000, 1, 1664, 1), (300, 9000, 1, 0, 1),        # more lists than units
    (0, 100, 3, 0, 3), (8, 100, 0, 0, 1)])
def test_whole_rounds_of_workgroups(lib, lists, rows, splits, cap, want):
    got = lib.kascade_decode_whole_rounds(lists, rows, splits, 256, cap)
    assert got == want
    if cap and lists and splits:
        assert rows / got <= max(cap, rows / splits)


def test_pooling_selects_where_the_rule_says(lib):
    """Prompt pooling: one launch or two, on both sides of each line."""
    from tests.test_gpu_prefill_units import POOLING_CASES, POOLING_CHUNKS
    calls = [(G, D, B, 0, L, want) for _, G, D, L, B, _, want in POOLING_CASES]
    calls += [(G, D, B, start, n, want) for _, G, D, start, n, B, want in POOLING_CHUNKS]
    assert {want for *_, want in calls} == {0, 1}
    for *call, want in calls:
        assert lib.kascade_prefill_pool_selects(*call) == want, call
    for none in ((0, 128, 1, 0, 32), (8, 128, 0, 0, 32), (8, 128, 1, 0, 0), (8, 128, 1, -32, 32), (8, 128, 1, 2 ** 31 - 32, 32)):
        assert lib.kascade_prefill_pool_selects(*none) == 0


def _err(lib):
    return lib.kascade_get_last_error().decode()


def test_sorted_topk_workspace_and_argument_checks(lib):
    import ctypes
    assert lib.kascade_topk_sorted_workspace_bytes(8192, 32768, 3328) == 0     # lists of up to 4096 entries: LDS
    assert (lib.kascade_topk_sorted_workspace_bytes(32, 524288, 52480)
            == (8 * 32 * 52480 + 255) // 256 * 256 + lib.kascade_topk_workspace_bytes(32, 524288))
    p = ctypes.c_void_p(256)
    assert lib.kascade_topk_sorted_call(p, p, 4, 10000, 10000, None, 1, 5000, None, None) == -1
    assert "workspace" in _err(lib)
    assert lib.kascade_topk_sorted_call(p, p, 4, 100, 100, None, 1, 101, p, None) == -1
    assert "k <= uniform_len" in _err(lib)


def test_null_pointers_are_rejected(lib):
    from kascade_amd._lib import Strides
    s = Strides(8, 8, 8)
    assert lib.kascade_decode_reuse_call(None, None, None, None, None, None, None, None, 1, 128, 128, 8, None, None) == -1
    assert "null pointer" in _err(lib)
    assert lib.kascade_decode_dense_paged_call(None, None, None, None, None, None, None, 1, 128, 8, None, 0, 16, None, None, None, None, None) == -1
    assert "null pointer" in _err(lib)
    assert lib.kascade_decode_recompute_paged_call(None, None, None, None, None, None, None, None, None, None,
                                                   1, 128, 128, 8, 1, None, 0, 16, None, None, None, None, None) == -1
    assert lib.kascade_topk_call(None, None, 1, 10, 10, None, None, 1, 4, 0, None, None) == -1
    assert lib.kascade_prefill_dense_call(None, None, None, None, None, 1, 64, s, s, 1, None) == -1
    assert lib.kascade_prefill_aggregate_call(None, None, None, None, 1, 64, s, s, 0, None) == -1
    assert lib.kascade_prefill_reuse_call(None, None, None, None, None, 10.0, None, 1, 64, 128, 1, s, s, None, None) == -1
    assert lib.kascade_paged_kv_append_call(None, None, None, None, None, None, 1, 1, 1, 16, s, None, None) == -1
    assert lib.kascade_rope_append_paged_call(None, None, None, None, None, None, 64, None, None, 1e-6, None, 0,
                                              None, None, None, None, 4, 16, 1, 1, None) == -1
    assert "null pointer" in _err(lib)


def test_bad_sizes_are_rejected(lib):
    from kascade_amd._lib import Strides
    buf = (C.c_char * 4096)()
    p = C.addressof(buf) & ~15          # fake, 16-byte aligned, never dereferenced: validation fails first
    p += 16
    assert lib.kascade_decode_reuse_paged_call(p, p, p, None, p, p, 0.0, p, p, p, 0, 128, 128, 8, None, 0, 16, None, None, None, None, None, None) == -1
    assert "batch" in _err(lib)
    assert lib.kascade_decode_reuse_paged_call(p, p, p, None, p, p, 10.0, p, p, p, 1, 128, 128, 8, None, 0, 16, None, None, None, None, None, None) == -1
    assert "cache_seqlens" in _err(lib)
    assert lib.kascade_decode_dense_paged_call(p, p, p, None, p, p, p, 1, 128, 8, p, 4, 12, None, None, None, None, None) == -1
    assert "power of two" in _err(lib)
    assert lib.kascade_decode_dense_paged_call(p + 2, p, p, None, p, p, p, 1, 128, 8, None, 0, 16, None, None, None, None, None) == -1
    assert "aligned" in _err(lib)
    hf = Strides(8 * 128 * 128, 128, 128 * 128)      # a head-major [B,G,L,D] cache seen as [B,L,G,D]
    assert lib.kascade_decode_dense_paged_call(p, p, p, None, p, p, p, 1, 128, 8, p, 4, 16, C.byref(hf), None, None, None, None) == -1
    assert "exclude each other" in _err(lib)
    assert lib.kascade_decode_dense_paged_call(p, p, p, None, p, p, p, 1, 128, 8, None, 0, 16,
                                               C.byref(Strides(1024, 4, 128)), None, None, None, None) == -1
    assert "strides" in _err(lib)
    assert lib.kascade_decode_dense_paged_call(p, p, p, None, p, p, p, 1, 128, 8, None, 0, 16, None, p, None, None, None) == -1
    assert "come together" in _err(lib)
    assert lib.kascade_decode_budgets_call(None, 1, 10.0, 1, None, None, None) == -1
    assert lib.kascade_decode_budgets_call(p, 1, 101.0, 1, None, None, None) == -1
    assert "topk_percent" in _err(lib)
    assert lib.kascade_topk_call(p, p, 4, 100, 200, None, None, 1, 8, 0, None, None) == -1
    assert "uniform_len" in _err(lib)
    assert lib.kascade_rope_append_paged_call(p, None, p, p, None, p, 64, None, None, 1e-6, p, 0, p, p, p, p,
                                              4, 12, 1, 1, None) == -1
    assert "power of two" in _err(lib)
    assert lib.kascade_rope_append_paged_call(p, C.byref(Strides(6144, 6140, 128)), p, p, None, p, 64, None, None,
                                              1e-6, p, 0, p, p, p, p, 4, 16, 1, 1, None) == -1
    assert "strides" in _err(lib)
    assert lib.kascade_rope_append_paged_call(p, None, p, p, None, p, 0, None, None, 1e-6, p, 0, p, p, p, p,
                                              4, 16, 1, 1, None) == -1
    assert "max_pos" in _err(lib)
    bad = Strides(100, 4, 128)          # not multiples of 8 elements
    ok = Strides(4096 * 128, 4096, 128)
    assert lib.kascade_prefill_dense_call(p, p, p, p, p, 1, 64, bad, ok, 1, None) == -1
    assert "strides" in _err(lib)
    assert lib.kascade_prefill_reuse_call(p, p, p, p, p, 0.0, p, 1, 64, 128, 1, ok, ok, None, None) == -1
    assert "rolling" in _err(lib)
    assert lib.kascade_prefill_reuse_call(p, p, p, p, p, 10.0, p, 1, 64, 0, 0, ok, ok, None, None) == -1
    assert "max_topk_num" in _err(lib)


def test_shape_descriptors_are_validated(lib):
    """Every *_shaped_call checks its kascade_shape before anything else."""
    from kascade_amd._lib import Shape, Strides
    buf = (C.c_char * 4096)()
    p = (C.addressof(buf) & ~15) + 16
    ok = Strides(4096 * 128, 4096, 128)
    rope = (p, None, p, p, None, p, 64, None, None, 1e-6, p, 0, p, p, p, p, 4, 16, 1, 1, None)
    chunk_dense = (p, p, p, p, p, 1, 0, 64, ok, p, 4, 16, 8, 1, None, None, None)
    budgets = (p, 1, 10.0, 1, None, None, None)
    for fn, args in ((lib.kascade_rope_append_paged_shaped_call, rope),
                     (lib.kascade_prefill_chunk_dense_shaped_call, chunk_dense),
                     (lib.kascade_decode_budgets_shaped_call, budgets)):
        assert fn(None, *args) == -1
        assert "shape" in _err(lib)
        assert fn(C.byref(Shape(8, 96, 0)), *args) == -1
        assert "head_dim" in _err(lib)
        assert fn(C.byref(Shape(0, 128, 0)), *args) == -1
        assert "kv_heads" in _err(lib)
        assert fn(C.byref(Shape(8, 128, 2)), *args) == -1
        assert "dtype" in _err(lib)
    # a valid shape reaches the argument checks of the call itself
    sh = C.byref(Shape(2, 64, 1))
    assert lib.kascade_prefill_chunk_dense_shaped_call(sh, p, p, p, p, p, 1, 16, 64, ok, p, 4, 16, 8, 1, None, None, None) == -1
    assert "multiple of 32" in _err(lib)
    assert lib.kascade_prefill_chunk_dense_shaped_call(sh, p, p, p, p, p, 1, 32, 64, ok, p, 8, 16, 8, 1, None, p, None) == -1
    assert "q_len_rows comes with q_start_rows" in _err(lib)
    assert lib.kascade_rope_append_paged_shaped_call(sh, p, None, p, p, None, p, 0, None, None, 1e-6, p, 0, p, p, p, p,
                                                     4, 16, 1, 1, None) == -1
    assert "max_pos" in _err(lib)
    assert lib.kascade_decode_budgets_shaped_call(sh, p, 1, 101.0, 1, None, None, None) == -1
    assert "topk_percent" in _err(lib)


def test_python_wrappers_fail_loudly_without_gpu():
    import torch
    from kascade_amd import kernels
    from kascade_amd._lib import KascadeError
    if torch.cuda.is_available():
        pytest.skip("GPU present")
    q = torch.zeros(1, 32, 128, dtype=torch.float16)
    with pytest.raises((KascadeError, RuntimeError)):
        kernels.decode_reuse(q, q, q, q, q, q, q)


def test_header_is_plain_c_and_links_from_c(lib, tmp_path):
    """The boundary is a C ABI: the header compiles as C99 (no C++ needed) and a C program
    linked against the library reads the ABI version and gets the error convention
    (-1 + message) without a GPU."""
    import shutil
    import subprocess
    from kascade_amd import _lib
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    src = tmp_path / "abi.c"
    src.write_text(
        '#include <stdio.h>\n#include <string.h>\n#include "kascade_hip.h"\n'
        "int main(void) {\n"
        "    if (kascade_abi_version() < 1) return 2;\n"
        "    if (kascade_topk_call(0, 0, 1, 10, 10, 0, 0, 1, 4, 0, 0, 0) != -1) return 3;\n"
        "    if (strlen(kascade_get_last_error()) == 0) return 4;\n"
        '    printf("%d\\n", kascade_abi_version());\n'
        "    return 0;\n}\n")
    exe = tmp_path / "abi"
    libdir = str(_lib.LIB_PATH.parent)
    subprocess.run([gcc, "-std=c99", "-Wall", "-Werror", "-pedantic", "-I", os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe), "-L", libdir, "-l:" + _lib.LIB_PATH.name,
                    "-Wl,-rpath," + libdir], check=True, capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True)
    assert int(out.stdout.strip()) == lib.kascade_abi_version()
