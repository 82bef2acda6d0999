"""The launch plans of csrc/gemm_plan.hpp and csrc/q32_plan.hpp as a host library."""
import ctypes
import functools
import os
import shutil
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include "q32_plan.hpp"
using namespace moe;
// 1: fine up kernel, 2: fine down kernel
extern "C" int fine(int64_t H, int64_t F, int64_t groups, int64_t k, int direct, int always_on, int64_t T) {
    const Q32Grid g = q32_grid(T, k, groups, direct != 0, always_on != 0);
    return q32_up_fine(F, g) + 2 * q32_down_fine(H, g);
}
extern "C" int tiled32(int64_t T, int64_t k, int64_t E) { return q32_tiled(T, k, E); }
// A tiled K-quant launch over `groups` lists: 1000 * tile + 10 * parts of K + (eight waves with rows of their own)
static int kernel(int dt, bool up, int64_t rows, int64_t k, int64_t slots, int64_t groups, int tile) {
    const GemmFormat f = gemm_format(dt);
    const int64_t tiles = max_gemm_tiles(slots, groups + 1, tile);
    const int parts = gemm_plan(f, up, rows, k, slots, groups, tile, tiles).parts;
    const bool one_operand = f.one_operand && !up && tile == 64;
    return 1000 * tile + 10 * parts + (parts == 1 && !one_operand && gemm_wide(up, rows, slots, groups, tile, tiles));
}
extern "C" int dense_kernel(int dt, int64_t n, int64_t k, int64_t m) {   // 0: streamed
    const int tile = gemm_dense_tile(gemm_format(dt), n, k, m);
    return tile == 0 ? 0 : kernel(dt, false, n, k, m, 1, tile);
}
extern "C" int up_kernel(int dt, int dt_down, int64_t H, int64_t F, int64_t T, int64_t k, int64_t E) {
    return kernel(dt, true, 2 * F, H, T * k, E, gemm_layer_plan(gemm_format(dt), gemm_format(dt_down), H, F, T, k, E).tile_slots);
}
extern "C" int down_kernel(int dt, int dt_down, int64_t H, int64_t F, int64_t T, int64_t k, int64_t E) {   // 0: streamed
    const LayerPlan lp = gemm_layer_plan(gemm_format(dt), gemm_format(dt_down), H, F, T, k, E);
    return lp.tiled_down ? kernel(dt_down, false, H, F, T * k, E, lp.tile_slots) : 0;
}
"""


@functools.lru_cache(None)
def load():
    """The library, or None without a host compiler."""
    gxx = shutil.which("g++")
    if gxx is None:
        return None
    d = tempfile.mkdtemp(prefix="plan")
    src, so = os.path.join(d, "plan.cpp"), os.path.join(d, "plan.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "candle_amd", "csrc"), src, "-o", so],
                   check=True)
    lib = ctypes.CDLL(so)
    shutil.rmtree(d)
    i64, i = ctypes.c_int64, ctypes.c_int
    lib.fine.argtypes = [i64, i64, i64, i64, i, i, i64]
    lib.tiled32.argtypes = [i64, i64, i64]
    lib.dense_kernel.argtypes = [i, i64, i64, i64]
    lib.up_kernel.argtypes = lib.down_kernel.argtypes = [i, i, i64, i64, i64, i64, i64]
    return lib
