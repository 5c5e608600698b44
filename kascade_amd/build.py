"""Builds libkascade_hip.so (gfx950) from kascade_amd/csrc with hipcc, and the extension module
_native (host code against torch's C++ interface, linked to that library) with g++.

Both are built in-tree (kascade_amd/libkascade_hip.so, kascade_amd/_native.so).  ``build()``
always recompiles; ``ensure_built()`` compiles only when no library exists.  The library needs hipcc
alone; without torch the extension, which only the Python strategies use, is left out, and without g++
ROCm's own clang builds it.
Run ``python -m kascade_amd.build`` to build from a shell.
"""
from __future__ import annotations

import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libkascade_hip.so"
NATIVE_PATH = PKG_DIR / "_native.so"
SOURCES = ["capi.hip", "decode.hip", "topk.hip", "prefill.hip", "paged.hip", "diag.hip"]
ARCH = "gfx950"

# -packed-fp32-ops is switched off for device code: hipcc otherwise forms
# v_pk_*_f32 from ordinary float code.  The host pass does not know the feature
# and prints a harmless warning.
COMMON_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
# The tile loops start on a 64-byte line of the instruction cache: where an edit happened to move them off it, a
# wavefront alone on its SIMD waited up to 90 cycles a round for its own instructions (log-sums alone, 8/2 heads of
# 64, 4096 tokens: 34.9 us, aligned 33.4, the same instructions).  The other sources' loops: no difference.
SOURCE_FLAGS = {"prefill.hip": ["-falign-loops=64"]}


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: libkascade_hip.so cannot be built")
    return exe


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines()
                    if "is not a recognized feature for this target" not in l)
    if proc.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(map(str, cmd)) + "\n" + out)
    return out


def build(verbose: bool = False, extra_flags=()) -> Path:
    hipcc = _hipcc()
    objdir = PKG_DIR / "build"
    objdir.mkdir(exist_ok=True)
    objs = []

    def compile_one(src):
        obj = objdir / (src + ".o")
        out = _run([hipcc, *COMMON_FLAGS, *SOURCE_FLAGS.get(src, ()), *extra_flags, "-c", str(CSRC / src), "-o", str(obj)])
        if verbose and out.strip():
            print(out)
        return obj

    with ThreadPoolExecutor(max_workers=min(4, len(SOURCES))) as ex:
        objs = list(ex.map(compile_one, SOURCES))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wno-unused-command-line-argument",
          *map(str, objs), "-o", str(tmp)])
    os.replace(tmp, LIB_PATH)
    if _torch_root() is None:
        print(f"torch is not installed: {LIB_PATH.name} is built, {NATIVE_PATH.name} (the Python strategies) is not")
    else:
        build_native()
    return LIB_PATH


def _torch_root():
    spec = importlib.util.find_spec("torch")
    return Path(spec.origin).resolve().parent if spec and spec.origin else None


def _host_compiler() -> str:
    return shutil.which("g++") or str(Path(_hipcc()).resolve().parent / "amdclang++")


def build_native() -> Path:
    """The host extension: plain C++ (no device code), so g++ builds it."""
    root = _torch_root()
    tmp = NATIVE_PATH.with_suffix(".so.tmp")
    _run([_host_compiler(), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", f"-I{root / 'include'}",
          f"-I{sysconfig.get_paths()['include']}", str(CSRC / "native.cpp"), f"-L{PKG_DIR}", "-l:libkascade_hip.so",
          f"-L{root / 'lib'}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-Wl,-rpath,$ORIGIN", "-o", str(tmp)])
    os.replace(tmp, NATIVE_PATH)
    return NATIVE_PATH


def ensure_built() -> Path:
    if not LIB_PATH.exists() or not (NATIVE_PATH.exists() or _torch_root() is None):
        build()
    return LIB_PATH


if __name__ == "__main__":
    path = build(verbose=True, extra_flags=sys.argv[1:])
    print(path)
