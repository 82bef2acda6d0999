"""The costs that choose a tiled K-quant product's slot tile and the parts its workgroups cut K into, as a program on the host:
the choices beside their lines, and that every choice is one the kernels exist for, over sizes of all orders."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "gemm_plan.hpp"
using namespace moe;
static GemmFormat fmt(int f) { return f == 0 ? GemmFormat{2.5, false, false, true} : f == 1 ? GemmFormat{5, true, true, false} : GemmFormat{5, true, false, false}; }
extern "C" int dense(int f, int64_t n, int64_t k, int64_t m) {   // 1000 * tile + parts; 0: streamed
    const int t = gemm_dense_tile(fmt(f), n, k, m);
    return t == 0 ? 0 : 1000 * t + gemm_plan(fmt(f), false, n, k, m, 1, t, max_gemm_tiles(m, 2, t)).parts;
}
extern "C" int layer(int f, int64_t H, int64_t F, int64_t slots, int64_t groups) {   // parts 0: the down projection streamed
    const LayerPlan lp = gemm_layer_plan(fmt(f), fmt(f), H, F, slots, groups);
    const int t = lp.tile_slots;
    const GemmPlan up = gemm_plan(fmt(f), true, 2 * F, H, slots, groups, t, max_gemm_tiles(slots, groups + 1, t));
    if (up.parts != 1) return -1;
    return 1000 * t + (lp.tiled_down ? gemm_plan(fmt(f), false, H, F, slots, groups, t, max_gemm_tiles(slots, groups + 1, t)).parts : 0);
}
"""
Q4K, Q5K, Q6K = 0, 1, 2


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
    lib.dense.argtypes = [ctypes.c_int, i64, i64, i64]
    lib.layer.argtypes = [ctypes.c_int, i64, i64, i64, i64]
    return lib


# us measured: streamed, one part, the choice
@pytest.mark.parametrize("f,n,k,m,want", [
    (Q4K, 4096, 4096, 384, 64002),     # 43.0, 36.8, 31.6
    (Q4K, 4096, 4096, 777, 128002),    # 77, 51.2, 45.4
    (Q4K, 4096, 4096, 4096, 128001),   # 321, 161; two parts 181
    (Q4K, 1024, 4096, 256, 0),         # 18.8; four parts 23.1
    (Q4K, 1024, 4096, 777, 64004),     # 28.2, 39, 27.8
    (Q4K, 14336, 4096, 128, 64002),    # 42, 47.4, 31.7
    (Q4K, 14336, 4096, 512, 128001),   # 142, 77.7; two parts 86.2
    (Q6K, 4096, 4096, 128, 0),         # 19.7; four parts 24.4
    (Q6K, 4096, 4096, 256, 64004),     # 29.9, 37, 26.9
    (Q6K, 4096, 14336, 1024, 128002),  # 314, 191, 155
    (Q5K, 4096, 4096, 777, 64001),     # 80.5, 61.8; two parts of 128 slots 66.0
    (Q4K, 4096, 4096, 95, 0),
    (Q4K, 4224, 4096, 95, 0),
    (Q4K, 4176, 4096, 777, 0),         # not a multiple of 128 rows
])
def test_dense_products(plan, f, n, k, m, want):
    assert plan.dense(f, n, k, m) == want


# the Mixtral shape and a quarter of its width, tokens; us per step before (streamed down projection or one part), and now
@pytest.mark.parametrize("f,H,F,tokens,want", [
    (Q4K, 4096, 14336, 137, 128002), (Q4K, 4096, 14336, 240, 128002), (Q4K, 4096, 14336, 301, 128002),   # 286 / 271, 395 / 323, 371 / 354
    (Q4K, 4096, 14336, 640, 128001), (Q4K, 4096, 14336, 3000, 128001),                                   # two parts 715 / 695, 2480 / 2507
    (Q6K, 4096, 14336, 200, 128002), (Q5K, 4096, 14336, 260, 128002), (Q5K, 4096, 14336, 777, 128001),   # 395 / 325, 547 / 408; 1021 / 903
    (Q6K, 1024, 3584, 137, 128000), (Q4K, 1024, 3584, 260, 128000),                                       # 50, four parts 52; 66 / 55, four parts 57
    (Q4K, 1024, 3584, 160, 64004), (Q4K, 1024, 3584, 500, 64002), (Q4K, 1024, 3584, 1000, 128002),       # 49 / 46, 103 / 76, 126 / 115
])
def test_routed_layers(plan, f, H, F, tokens, want):
    assert plan.layer(f, H, F, 2 * tokens, 8) == want


def test_every_choice_has_a_kernel(plan):
    for f in (Q4K, Q5K, Q6K):
        for n in (128, 256, 384, 512, 1152, 4096, 14336, 65536):
            for k in (256, 512, 768, 1280, 4096, 14336):
                for m in (1, 95, 96, 113, 128, 129, 300, 777, 2049, 60000):
                    assert plan.dense(f, n, k, m) in (0, 64001, 64002, 64004, 128001, 128002), (f, n, k, m)
        for H, F in ((128, 256), (768, 512), (1024, 3584), (4096, 14336)):
            for E in (1, 2, 8, 60, 256):
                for per in (35, 64, 100, 129, 1000):
                    assert plan.layer(f, H, F, per * E, E) in (64000, 64001, 64002, 64004, 128000, 128001, 128002), (f, H, F, E, per)
