"""The planner's estimates (csrc/gdn_plan_model.h), compiled for the host, against
measured times: for each batch the call was timed at every segment length
(MI355X, near-1 decay, us per call), and the length of the smallest estimate
must be within 5% of the fastest (the timings repeat to 2%)."""

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "kachua_mlsys_amd" / "csrc"
WHOLE = 1 << 30

SHIM = """
#include "gdn_plan_model.h"
extern "C" float split_mrun_us(float chunks, float first, float segments, float longs, float shorts, float mfrac,
                               int longest, int L) {
  return gdn::plan_split_mrun_us(gdn::PlanStats{chunks, first, segments, longs, shorts, mfrac, longest, L});
}
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    cxx = shutil.which("c++") or shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("plan_model")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(d / "shim.cpp"), "-o",
                    str(d / "shim.so")], check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    lib.split_mrun_us.restype = ctypes.c_float
    lib.split_mrun_us.argtypes = [ctypes.c_float] * 6 + [ctypes.c_int] * 2
    return lib


def _stats(lengths, L):
    n = [(x + 63) // 64 for x in lengths]
    longs = [c for c in n if c >= 2]
    return (sum(longs), sum(min(c, L) for c in longs), sum((c - 1) // L + 1 for c in longs), len(longs),
            len(n) - len(longs), 1.0, max(longs), L)


# lengths -> {segment length in chunks (0: whole sequences): us per call}
SPLIT = {
    "1 x 2000": ([2000], {4: 62.9, 6: 58.9, 8: 53.4, 10: 56.2, 12: 59.0, 16: 62.5, 0: 82.3}),
    "1 x 8192": ([8192], {8: 124.6, 10: 123.2, 12: 126.5, 16: 95.1, 20: 98.5, 32: 109.5, 64: 164.4, 0: 278.9}),
    "1 x 32768": ([32768], {16: 309.4, 22: 278.3, 32: 246.3, 48: 297.1, 64: 232.9, 80: 262.0, 128: 341.9, 0: 1068.9}),
    "2 x 1000": ([919, 1081], {4: 53.7, 6: 49.0, 8: 50.9, 10: 48.9, 12: 52.1, 16: 56.8, 0: 53.3}),
    "4 x 2000": ([910, 2170, 2731, 2189], {4: 109.9, 8: 92.7, 12: 82.2, 14: 72.7, 16: 75.7, 20: 79.0, 32: 94.4, 0: 107.3}),
    "8 x 1000": ([835, 1092, 900, 708, 846, 1599, 996, 1024],
                 {6: 87.4, 8: 80.2, 10: 72.1, 12: 63.7, 14: 60.0, 16: 60.7, 20: 67.9, 24: 74.5, 0: 71.4}),
    "16 x 1024": ([808, 1345, 1651, 661, 1653, 1437, 1442, 739, 1333, 1185, 714, 634, 615, 683, 540, 944],
                  {8: 123.0, 12: 97.5, 16: 88.3, 20: 74.8, 22: 76.7, 24: 78.7, 0: 75.9}),
    "1900 among 31 ones": ([1900] + [1] * 31, {4: 67.2, 6: 62.0, 8: 53.8, 10: 56.0, 12: 59.8, 16: 60.5, 28: 83.2, 0: 80.4}),
}


@pytest.mark.parametrize("name", list(SPLIT))
def test_split_mrun_segment_length(model, name):
    lengths, times = SPLIT[name]
    chosen = min(times, key=lambda L: (model.split_mrun_us(*_stats(lengths, L or WHOLE)), -(L or WHOLE)))
    assert times[chosen] <= 1.05 * min(times.values()), f"{name}: chose {chosen}, {times}"
