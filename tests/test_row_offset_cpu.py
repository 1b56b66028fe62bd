"""The masked decode's row offsets (csrc/ck_row_offset.h) in heads close to 2^31
bytes, compiled with g++: never past the last row."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "carrykernel_amd", "csrc")

SOURCE = r"""
#include "ck_row_offset.h"
// rows around the end of the largest head of K bytes a row that the entry point
// takes (V K < 2^31), one or more rows a lane: the number of wrong offsets
extern "C" int64_t wrong_offsets(int K) {
  const int V = (int)((((int64_t)1 << 31) - 1) / K);
  int64_t wrong = 0;
  for (int64_t r = V - 8; r < V + 2048; ++r)
    for (int step = 0; step <= 192; step += 64) {
      if (r + step > 0x7fffffff) continue;
      const int64_t want = (r + step < V ? r + step : V - 1) * (int64_t)K;
      wrong += (int64_t)ck::pd::clamped_row_offset((int)r, step, K, V) != want;
    }
  return wrong;
}
"""


@pytest.mark.parametrize("K", [5, 17, 18, 44, 100, 257, 1000, 1023])
def test_rows_past_the_head_are_clamped(K, tmp_path):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, so = tmp_path / "rows.cpp", tmp_path / "rows.so"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.wrong_offsets.restype = ctypes.c_int64
    assert lib.wrong_offsets(K) == 0
