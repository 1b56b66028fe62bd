"""The size of one launch (csrc/ck_launch.h), compiled with g++: fewer than 2^32
work items, and slices that cover everything once."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "carrykernel_amd", "csrc")

SOURCE = r"""
#include "ck_launch.h"
// launches of n parts, 0 where they do not cover 0 .. n - 1 in order or one is
// too large (a part of more workgroups than a launch holds goes alone)
extern "C" int64_t launches(int64_t n, int64_t per_part, int threads) {
  int64_t next = 0, count = 0;
  const int status = ck::launch_slices(n, per_part, threads, [&](int64_t i, int64_t c) {
    if (i != next || c < 1 || (c > 1 && c * per_part * threads >= ((int64_t)1 << 32))) return 1;
    next = i + c;
    ++count;
    return 0;
  });
  return status == 0 && next == n ? count : 0;
}
"""


@pytest.mark.parametrize("n,per_part,threads,expect", [
    (1, 1, 64, 1), ((1 << 24) - 1, 1, 256, 1), (1 << 24, 1, 256, 2), ((1 << 24) + 5, 1, 256, 2),
    (1 << 22, 4, 256, 2), ((1 << 22) - 1, 4, 256, 1), (3, 1 << 24, 256, 3), (100000, 40961, 320, 306)])
def test_slices(n, per_part, threads, expect, tmp_path):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, so = tmp_path / "launch.cpp", tmp_path / "launch.so"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.launches.restype = ctypes.c_int64
    lib.launches.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    assert lib.launches(n, per_part, threads) == expect
