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
extern "C" int memory(long long rows, long long cols, int nk, int cus) { return tgx::line_share_tile(rows, cols, nk, cus); }
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


# what a step asks for covers every product that it bounds: 256 x 256 tiles are taken from more than two rounds of 128 x 128 on (tile_of: 28 to 10), and a smaller one needs the smaller tile
@pytest.mark.parametrize("cus", [8, 64, 256])
def test_memory_covers_every_product(plan, cus):
    up = lambda a, b: -(-a // b)      # noqa: E731
    for rows in [65, 128, 129, 1000, 2048, 4161]:
        for cols in [64, 320, 1024, 2048, 12416]:
            for nk in [1, 15, 16, 31, 32, 97]:
                for m in {min(65, rows), min(128, rows), rows // 2 + 1, rows}:
                    for n in {64, cols // 2, cols}:
                        t256, t128 = up(m, 256) * up(n, 256), up(m, 128) * up(n, 128)
                        tile = 256 if up(t256, cus) * 28 <= up(t128, cus) * 10 else 128
                        if plan.halved(t256 if tile == 256 else t128, tile, nk, cus):
                            assert plan.memory(rows, cols, nk, cus) >= tile, (rows, cols, nk, m, n)
