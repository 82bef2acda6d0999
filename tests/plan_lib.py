"""The launch plans of csrc/q32_plan.hpp as a host library."""
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
extern "C" int fine(int64_t H, int64_t F, int64_t groups, int64_t k, int direct, int always_on, int tiles, int64_t T) {
    const Q32Grid g = q32_grid(T, k, groups, direct != 0, always_on != 0);
    return q32_up_fine(F, g, tiles) + 2 * q32_down_fine(H, g);
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
    lib.fine.argtypes = [i64, i64, i64, i64, i, i, i, i64]
    return lib
