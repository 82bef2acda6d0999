"""The rule that gives a tiled K-quant launch workgroups of eight or of four waves, as a program on the host: the widths that
measured faster at the sizes next to its lines, and what it counts the workgroups of an XCD by."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "gemm_plan.hpp"
using namespace moe;
extern "C" int wide(int up, int64_t rows, int64_t slots, int64_t groups, int tile) {
    return gemm_wide(up != 0, rows, slots, groups, tile, max_gemm_tiles(slots, groups + 1, tile));
}
extern "C" int64_t busiest(int64_t n_rb, int64_t tiles, int64_t max_tiles) { return busiest_xcd(n_rb, tiles, max_tiles); }
// the same from the kernel's own walk over workgroup ids; -1: a pair of row block and tile that is not visited once
extern "C" int64_t walked(int64_t n_rb, int64_t tiles, int64_t max_tiles) {
    const int patch = patch_edge(n_rb, max_tiles), grid = (int)patch_grid(n_rb, max_tiles, patch);
    int64_t n[8] = {0}, seen = 0, key = 0;
    for (int b = 0; b < grid; b++) {
        const PatchPos p = patch_position(b, (int)n_rb, patch);
        if (p.tile >= tiles || p.rblk >= n_rb) continue;
        n[b & 7]++; seen++; key += p.tile * n_rb + p.rblk;
    }
    const int64_t all = n_rb * tiles;
    return seen == all && key == all * (all - 1) / 2 ? *std::max_element(n, n + 8) : -1;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("plan")
    src, so = d / "plan.cpp", d / "plan.so"
    src.write_text(SOURCE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "candle_amd", "csrc"), str(src),
                    "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    i64 = ctypes.c_int64
    lib.wide.argtypes = [ctypes.c_int, i64, i64, i64, ctypes.c_int]
    for f in (lib.busiest, lib.walked):
        f.argtypes, f.restype = [i64, i64, i64], i64
    return lib


# (weight rows, activation rows, slots per tile) of dense products; rounds of the busiest XCD, wide / narrow, and us of Q4_K
@pytest.mark.parametrize("n,m,tile,wide", [
    (4096, 512, 64, 0),      # 0.5: 46.5 wide / 38.6 narrow
    (4096, 576, 64, 1),      # 0.56: 47.4 / 51.3
    (4096, 777, 64, 1),      # 1.0 / 0.81: 51.0 / 52.8
    (4096, 1024, 64, 1),     # 1.0: 52.3 / 55.6
    (14336, 300, 64, 0),     # 1.25 / 1.19: 79.6 / 70.4
    (14336, 192, 64, 1),     # 0.75: 45.6 / 48.9
    (14336, 512, 64, 1),     # 2.0: 90.5 / 95.0
    (4096, 1500, 64, 1),     # 1.5 / 2.0: 89.4 / 96.0
    (4096, 2200, 128, 0),    # 1.25 / 1.12: 143 / 120
    (4096, 2800, 128, 0),    # 1.5 / 1.38: 150 / 130
    (4096, 3000, 128, 1),    # 1.5 / 2.0: 152 / 161
    (4096, 4096, 128, 1),    # 2.0: 159 / 162
    (14336, 1100, 128, 0),   # 2.25: 193 / 177
    (14336, 1450, 128, 1),   # 3.0: 221 / 227
    (14336, 1664, 128, 0),   # 3.12 / 3.25: 282 / 258
    (32000, 300, 128, 1),    # 1.5: 105 / 125
    (32000, 512, 128, 1),    # 2.0: 152 / 157
    (32000, 640, 128, 0),    # 2.5: 211 / 193
    (512, 16384, 128, 0),    # 187 / 138: too few row blocks
    (768, 16384, 128, 1),    # 191 / 195
    (4224, 1024, 64, 0),     # not a multiple of 256 rows
])
def test_dense_products(plan, n, m, tile, wide):
    assert plan.wide(0, n, m, 1, tile) == wide


# Mixtral shape (eight experts, top-2), tokens and slots per tile: the up projection (w1 and w3), the down projection
@pytest.mark.parametrize("tokens,tile,up,down", [
    (137, 64, 0, 0), (200, 64, 0, 0), (257, 64, 0, 1), (301, 128, 1, 0), (400, 128, 1, 0), (450, 128, 1, 0), (500, 128, 0, 1),
    (600, 128, 0, 1), (873, 128, 0, 1), (1000, 128, 0, 0), (2048, 128, 1, 0), (4096, 128, 1, None),
])
def test_routed_layers(plan, tokens, tile, up, down):
    assert plan.wide(1, 2 * 14336, 2 * tokens, 8, tile) == up
    assert down is None or plan.wide(0, 4096, 2 * tokens, 8, tile) == down


def test_workgroups_of_the_busiest_xcd(plan):
    for n_rb in (1, 2, 7, 16, 33, 56, 125, 224):
        for tiles in (1, 2, 3, 5, 8, 13, 19, 40):
            for spare in (0, 2, 9):
                assert plan.busiest(n_rb, tiles, tiles + spare) == plan.walked(n_rb, tiles, tiles + spare), (n_rb, tiles, spare)
