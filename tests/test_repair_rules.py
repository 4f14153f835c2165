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
    for units in (1, 255, 256, 640, 1792, 100000):
        t = rules.r_grad_tile(units, wd, 256)
        assert -(-wd // cols[t]) * cols[t] * 19 <= least * 20, (units, t)
        if wd % 128 == 0 and 2 * units * (wd // 128) >= 5 * 256:
            assert t == 0
        if units >= 256 and wd <= 64:
            assert t == (3 if wd <= 32 else 1)
