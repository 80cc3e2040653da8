"""How a prompt's products are cut (tinygpt_amd/csrc/prefill_plan.h): the rules are arithmetic on sizes, compiled here with the host compiler and gone through without a GPU."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

SOURCE = r"""
#include "prefill_plan.h"
// the first product (columns n, K, rows m) that is cut so that a slab holds no K: 1 and its sizes in out, 0: none
extern "C" int empty_slab(int cus, int k_lo, int k_hi, int* out) {
  for (int k = k_lo; k < k_hi; k += 64)
    for (int n = 64; n <= 8192; n += 64)
      for (int m = 129; m <= 1500; m += m < 260 ? 4 : 41) {
        const int z = tgx::eight_wave_slabs(m, n, k, cus), per = 64 * tgx::slab_steps(k, z);
        if (z < 1 || z > 8 || (z > 1 && (z - 1) * per >= k) || z * per < k) { out[0] = m; out[1] = n; out[2] = k; out[3] = z; return 1; }
      }
  return 0;
}
extern "C" int whole(int m, int n, int k, int cus, int most) { return tgx::gate_up_whole(m, n, k, cus, most); }
extern "C" int slabs(int m, int n, int k, int cus) { return tgx::eight_wave_slabs(m, n, k, cus); }
extern "C" int halves(int stages) { return tgx::eight_wave_halves(stages); }
extern "C" int steps(int k, int z) { return tgx::slab_steps(k, z); }
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, lib = d / "plan.cpp", d / "libplan.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "tinygpt_amd", "csrc"), str(src), "-o", str(lib)])
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("cus", [64, 256, 304])
@pytest.mark.parametrize("k_lo,k_hi", [(64, 2048), (2048, 4096), (4096, 16448)])
def test_no_slab_is_empty(plan, cus, k_lo, k_hi):
    """an empty slab's workgroups have nothing to wait for and nothing to add: the kernel counts on K in each of them"""
    out = (ctypes.c_int * 4)()
    assert plan.empty_slab(cus, k_lo, k_hi, out) == 0, dict(zip(("rows", "columns", "K", "slabs"), out))


@pytest.mark.parametrize("rows,columns,K,slabs", [(129, 1600, 1600, 5), (245, 1600, 1600, 5), (200, 1856, 1856, 6), (133, 2048, 2048, 8), (509, 1024, 2048, 5), (300, 2048, 8192, 5), (2048, 2048, 2048, 1)])
def test_slabs_of_products(plan, rows, columns, K, slabs):
    z = plan.slabs(rows, columns, K, 256)
    assert z == slabs
    assert (z - 1) * plan.steps(K, z) < K // 64 <= z * plan.steps(K, z)


# (rows, tiles of 128 columns, K): a short K from a quarter of a chip of 256 on, any from more than half a chip on; never at rows that the slabs' 64-row tiles fit
@pytest.mark.parametrize("rows,column_tiles,K,whole", [(133, 48, 1024, 1), (129, 32, 1024, 1), (129, 31, 1024, 0), (129, 32, 1088, 0), (128, 64, 1024, 0), (128, 129, 1024, 1), (133, 76, 896, 1),
                                                       (509, 48, 1024, 1), (100, 128, 3072, 0), (129, 64, 3072, 0), (129, 65, 3072, 1), (65, 224, 4096, 1), (64, 224, 4096, 0), (100, 256, 3072, 0), (300, 96, 1024, 0)])
def test_gate_up_whole(plan, rows, column_tiles, K, whole):
    assert plan.whole(rows, 128 * column_tiles, K, 256, 8) == whole
    assert plan.whole(rows, 128 * column_tiles - 2, K, 256, 8) == whole


def test_gate_up_is_whole_only_where_the_eight_wave_kernel_takes_it(plan):
    """the product is left without slabs for that kernel alone (prefill.wide_8k_max: its tiles in half-chips)"""
    for most in (0, 1, 2, 8):
        for tiles in range(1, 300):
            assert not (plan.whole(100, 128 * tiles, 512, 256, most) and 2 * tiles > most * 256)
    assert not plan.whole(133, 128 * 48, 1024, 256, 0) and plan.whole(133, 128 * 48, 1024, 256, 1)


def test_short_chains_of_stages_are_halved(plan):
    assert [plan.halves(n) for n in (1, 4, 32, 33, 128)] == [1, 1, 1, 0, 0]


@pytest.mark.parametrize("rows,columns,K,slabs", [(384, 1024, 3072, 8), (385, 1024, 3072, 7), (509, 1024, 3072, 5), (600, 1024, 3072, 5), (509, 896, 4864, 8)])
def test_slabs_of_more_than_three_row_tiles(plan, rows, columns, K, slabs):
    assert plan.slabs(rows, columns, K, 256) == slabs
