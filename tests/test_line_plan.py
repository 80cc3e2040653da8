"""How the last tiles of a prompt's product are divided (tinygpt_amd/csrc/line_plan.h): arithmetic on sizes, compiled with the host compiler and gone through without a GPU."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

SOURCE = r"""
#include "line_plan.h"
// 0: whole rounds first, then at most half a round of tiles as two halves that hold K together; otherwise what is wrong
extern "C" int walk(int tiles, int tile, int nk, int cus) {
  const tgx::LineShare s = tgx::line_share(tiles, tile, nk, cus);
  if (s.whole + s.rest != tiles || s.rest < 0) return 1;
  if (s.rest && (s.whole % cus || 2 * s.rest > cus || nk / 2 < 8)) return 2;
  return 0;
}
extern "C" int halved(int tiles, int tile, int nk, int cus) { return tgx::line_share(tiles, tile, nk, cus).rest; }
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("line")
    src, lib = d / "plan.cpp", d / "libplan.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "tinygpt_amd", "csrc"), str(src), "-o", str(lib)])
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("cus", [1, 8, 64, 255, 256, 304])
@pytest.mark.parametrize("tile", [128, 256])
def test_rounds_and_halves(plan, tile, cus):
    for nk in [1, 2, 15, 16, 17, 31, 32, 33, 97, 256]:
        for tiles in range(0, 3 * cus + 2):
            assert plan.walk(tiles, tile, nk, cus) == 0, (tiles, nk, cus)


@pytest.mark.parametrize("tiles,tile,nk,halved", [(344, 256, 128, 88), (344, 256, 16, 88), (344, 256, 15, 0), (256, 256, 128, 0), (384, 128, 32, 128), (385, 128, 32, 0), (384, 128, 31, 0), (1, 128, 64, 1)])
def test_what_is_halved(plan, tiles, tile, nk, halved):
    assert plan.halved(tiles, tile, nk, 256) == halved
