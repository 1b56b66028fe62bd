"""The statequant kernels' split of V columns over workgroups (csrc/ck_tiles.h,
host code), compiled by itself with g++ and enumerated."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "carrykernel_amd", "csrc")

# bad_tiles: the first V of lo..hi whose tiles are not as TileForm says (0: none)
SOURCE = r"""
#include "ck_tiles.h"
using namespace ck::qs;
static bool good(int64_t V, int KP, bool fp32_rows, bool ingest) {
  const ColTiles t = col_tiles((int)V, KP, fp32_rows, ingest);
  const int S = KP <= 128 ? 8 : KP / 16, cpt = t.form == kTileOne ? 1 : 4;
  const int64_t last = V - (int64_t)(t.nvt - 1) * t.width;  // columns of the last tile
  if (t.nvt < 1 || t.width != t.groups * cpt || last < 1 || last > t.width) return false;
  const bool reach = ingest ? V <= 1 << 30 : KP * V < (int64_t)1 << 32;
  if (t.form == kTileOne) return t.groups == kGroups && (V < 4 || !reach);
  if (!reach) return false;
  if (last < 4 || V < 4) return false;                      // no column of another workgroup's
  if (t.form == kTileFull) return t.groups == kGroups && V % 4 == 0;
  return t.groups >= 1 && t.groups <= max_groups(KP) && tile_threads(t, S) <= max_groups(KP) * S;
}
extern "C" int64_t bad_tiles(int64_t lo, int64_t hi, int KP, int fp32_rows, int ingest) {
  for (int64_t V = lo; V <= hi; ++V)
    if (!good(V, KP, fp32_rows != 0, ingest != 0)) return V;
  return 0;
}
extern "C" int bad_inverse() {
  for (uint32_t g = 1; g <= 40; ++g)
    for (uint32_t x = 0; x < 1024; ++x)
      if ((x * ((65536u + g - 1) / g)) >> 16 != x / g) return (int)(g * 1024 + x);
  return 0;
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("tiles")
    src, so = d / "tiles.cpp", d / "tiles.so"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.bad_tiles.restype = ctypes.c_int64
    lib.bad_tiles.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    return lib


@pytest.mark.parametrize("KP", [16, 128, 256])
@pytest.mark.parametrize("fp32_rows", [0, 1])
@pytest.mark.parametrize("ingest", [0, 1])
def test_no_tile_reaches_into_another(rules, KP, fp32_rows, ingest):
    """The last tile keeps 4 columns, so no thread is moved into another
    workgroup's columns (V = 6241 at K <= 128 and 3969 at K > 128 once did)."""
    assert rules.bad_tiles(1, 1 << 22, KP, fp32_rows, ingest) == 0
    limit = 1 << 30 if ingest else (1 << 32) // KP
    assert rules.bad_tiles(limit - 4096, limit + 4096, KP, fp32_rows, ingest) == 0


def test_group_division(rules):
    assert rules.bad_inverse() == 0
