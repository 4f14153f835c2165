"""The host rules that choose phase 2's kernels (csrc/repair_rule.h), compiled with the host compiler."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cdcl-gptq_amd", "csrc")
SHIM = """
#include "repair_rule.h"
using namespace cdclq;
extern "C" {
int r_grad_tile(long units, int wd, int cus) { return (int)grad_tile(units, wd, cus); }
int r_share_rounds(int grid, int units) {  // every unit once; returns the most that one workgroup takes
  const int nx = grid < 8 ? grid : 8;
  int next = 0, most = 0;
  for (int x = 0; x < nx; ++x) {
    const GradShare s = grad_share(x, grid, nx, units);
    if (s.first != next || s.stride != (grid - x + nx - 1) / nx) return -1;
    next = s.end;
    const int r = (s.end - s.first + s.stride - 1) / s.stride;
    most = r > most ? r : most;
  }
  return next == units ? most : -1;
}
int r_cd_panel_ok(int n, int sbw, int rows, int cus) { return cd_panel_ok(n, sbw, rows, cus); }
int r_cd_panel_pays(const int* tiles, int nsub, int both, int np, int rows, int sweeps, int cus) {
  return cd_panel_pays(tiles, nsub, both, np, rows, sweeps, cus);
}
int r_refit_panel_ok(int n, int g, int rows, int cus) { return refit_panel_ok(n, g, rows, cus); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(d / "shim.cpp"),
                    "-o", str(d / "shim.so")], check=True)
    L = C.CDLL(str(d / "shim.so"))
    L.r_grad_tile.argtypes = [C.c_long, C.c_int, C.c_int]
    return L


@pytest.mark.parametrize("wd", [4, 8, 16, 32, 48, 60, 64, 68, 96, 100, 128, 192, 196, 256, 320, 512, 1000, 1024])
def test_gradient_tile_computes_few_spare_columns(rules, wd):
    """The 128-column tile computes at most 1/19 more columns than 64-column ones would, and is still taken
    for widths that it divides once it fills the device; 32 columns and fewer take the 32-column tile there."""
    cols = {0: 128, 1: 64, 2: 64, 3: 32}
    least = (wd + 63) // 64 * 64
    for units in (1, 128, 255, 256, 640, 1792, 100000):
        t = rules.r_grad_tile(units, wd, 256)
        assert -(-wd // cols[t]) * cols[t] * 19 <= least * 20, (units, t)
        if wd % 128 == 0 and 2 * units * (wd // 128) >= 5 * 256:
            assert t == 0
        if units >= 256 and wd <= 64:
            assert t == (3 if wd <= 32 else 1)
        if units <= 128 and wd <= 64:
            assert t == 2


def test_gradient_units_spread_over_the_workgroups(rules):
    """A workgroup per unit is one round, whatever the count is modulo the XCDs; more units take one round
    more than their share at most."""
    for units in [*range(1, 300), 511, 767, 768]:
        assert rules.r_share_rounds(min(units, 768), units) == 1, units
    for units in (769, 1000, 1535, 1536, 5000, 24640):
        assert -(-units // 768) <= rules.r_share_rounds(768, units) <= -(-units // 768) + 1, units


@pytest.mark.parametrize("n,g,most", [  # the most rows on 256 CUs; None: any number
    (2048, 128, 8192), (6144, 128, 8192), (6145, 128, 4096), (128, 128, 8192), (100, 100, 8192), (65, 65, 8192),   # two pieces to a group
    (64, 64, 16384), (20, 20, 16384),                                        # one group, one piece
    (65, 64, None), (2048, 64, None), (2048, 32, None), (300, 16, None),     # groups inside a piece
    (2048, 8, 0), (2048, 96, 0), (2048, 256, 0), (300, 300, 0), (2048, 24, 0),
])
def test_refit_by_panels(rules, n, g, most):
    """Groups that fit the panels' pieces take the panel launch while their rows are few rounds of it."""
    for rows in (1, 4096, 4097, 8192, 8193, 16384, 16385, 1 << 20):
        assert rules.r_refit_panel_ok(n, g, rows, 256) == (most is None or rows <= most), rows


@pytest.mark.parametrize("n,sub_block,most", [(64, 64, 12288), (64, 100, 12288), (40, 40, 12288), (128, 64, 12288),
                                              (129, 64, 24576), (512, 64, 24576), (513, 64, None), (4096, 64, None),
                                              (128, 128, 0), (4096, 48, 0), (65, 65, 0)])
def test_descent_by_panels(rules, n, sub_block, most):
    for rows in (1, 12288, 12289, 24576, 24577, 1 << 20):
        assert rules.r_cd_panel_ok(n, sub_block, rows, 256) == (most is None or rows <= most), rows


@pytest.mark.parametrize("rows", [1, 256, 1024, 4096, 14336, 32768, 131072])
@pytest.mark.parametrize("np_", [3, 4, 16, 56])
def test_descent_panels_of_a_sparse_selection(rules, rows, np_):
    """A panel whose four sub-blocks every tile selected is one launch; one of them alone, or from 8192 rows on
    two, take a launch each; of many panels also four that a quarter of the tiles each selected, whose spare
    columns cost more than three launches."""
    cus, tiles = 256, -(-rows // 128)

    def pays(t, both, sweeps=1):
        return rules.r_cd_panel_pays((C.c_int * len(t))(*t), len(t), both, np_, rows, sweeps, cus)

    assert pays([tiles] * 4, tiles)
    if rows <= 14336 or np_ > 16:
        assert pays([tiles] * 4, tiles, 2)  # two sweeps: at few panels not from many rounds of rows on
    elif rows > 32768 and np_ <= 4:
        assert not pays([tiles] * 4, tiles, 2)
    assert not pays([0, 0, tiles, 0], tiles)
    if rows > 8192:
        assert not pays([tiles, 0, tiles, 0], tiles)
        if np_ >= 16:
            assert not pays([tiles // 4] * 4, tiles)


def test_descent_of_one_panel_needs_no_gradient(rules):
    assert rules.r_cd_panel_pays((C.c_int * 4)(0, 1, 0, 0), 4, 1, 1, 4096, 1, 256)
