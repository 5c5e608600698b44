"""The prefill kernels' own budget arithmetic (csrc/budgets.h), compiled for the host: it decides for every unit
between dense and sparse and how far its list is read, and has to agree with what the host sizes lists by."""
import ctypes
import subprocess

import numpy as np
import pytest

from kascade_amd import budgets, build

STARTS = np.arange(0, (1 << 20) + 1, 32, dtype=np.int32)   # a prompt's tiles, up to a million tokens


@pytest.fixture(scope="module")
def device_budgets(tmp_path_factory):
    out = tmp_path_factory.mktemp("budgets")
    (out / "b.cpp").write_text("""
#define __host__
#define __device__
#include "budgets.h"
extern "C" void rolling(float pct, const int* at, int n, int* out) {
    for (int i = 0; i < n; ++i) out[i] = kascade::rolling_budget(pct, at[i]);
}
extern "C" void width(float pct, const int* at, int n, int* out) {
    for (int i = 0; i < n; ++i) out[i] = kascade::topk_width_of(pct, at[i]);
}
""")
    subprocess.run([build._host_compiler(), "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{build.CSRC}", str(out / "b.cpp"),
                    "-o", str(out / "b.so")], check=True, capture_output=True)
    lib = ctypes.CDLL(str(out / "b.so"))

    def call(name, pct, at):
        res = np.empty(len(at), np.int32)
        as_ints = ctypes.POINTER(ctypes.c_int)
        getattr(lib, name)(ctypes.c_float(pct), at.ctypes.data_as(as_ints), len(at), res.ctypes.data_as(as_ints))
        return res
    return call


def _rounded_up(entries):
    return (np.maximum(entries, 128) + 127) // 128 * 128


@pytest.mark.parametrize("pct", [0.01, 0.1, 0.7, 1, 3.3, 5, 7, 10, 12.5, 12.7, 20, 33, 33.3, 50, 66.6, 99.9, 100])
def test_rolling_budget_is_the_floor_of_the_quotient(device_budgets, pct):
    """Every tile start, as the quotient gives it in float64 and, for whole percentages, in whole numbers (starts
    where pct start is a multiple of 100 among them), and as the host counts lists."""
    got = device_budgets("rolling", pct, STARTS)
    quotient = np.floor(np.float64(np.float32(pct)) * STARTS.astype(np.float64) / 100.0).astype(np.int64)
    assert np.array_equal(got, _rounded_up(quotient))
    if float(pct).is_integer():
        assert np.array_equal(got, _rounded_up(int(pct) * STARTS.astype(np.int64) // 100))
        assert all(budgets.rolling_budget(int(s), pct) == g for s, g in zip(STARTS[::97], got[::97]))


@pytest.mark.parametrize("pct", [100.5, 1e3, 4e5, 1e6, 1e7, 1e12, 3e38, float("inf")])
def test_percentages_above_100_take_the_whole_list(device_budgets, pct):
    """The reuse calls take any percentage: what it asks for beyond a tile's own keys is cut to the list's width by
    the caller and must not wrap around on the way."""
    at = STARTS[1:]
    got = device_budgets("rolling", pct, at)
    assert (got >= at).all() and (got % 128 == 0).all()


@pytest.mark.parametrize("pct", [1, 5, 10, 12.5, 33, 100])
def test_row_width_is_the_hosts(device_budgets, pct):
    at = np.unique(np.concatenate([np.arange(1, 3000), STARTS[1::61]])).astype(np.int32)
    assert np.array_equal(device_budgets("width", pct, at), [budgets.topk_width(int(L), pct) for L in at])
