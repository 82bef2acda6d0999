"""The rule that gives a tiled K-quant launch workgroups of eight or of four waves, as a program on the host: the widths that
measured faster at the sizes next to its lines."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def gemm_wide(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("plan")
    src, so = d / "plan.cpp", d / "plan.so"
    src.write_text('#include "gemm_plan.hpp"\nextern "C" int wide(int up, int64_t rows, int64_t slots, int64_t groups, int tile)\n'
                   '{ return moe::gemm_wide(up != 0, rows, slots, groups, tile); }\n')
    subprocess.run([gxx, "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "candle_amd", "csrc"), str(src), "-o", str(so)], check=True)
    f = ctypes.CDLL(str(so)).wide
    f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return f


# (weight rows, activation rows, slots per tile) of dense products: wide, with the rounds of 256 wide workgroups in the comment
@pytest.mark.parametrize("n,m,tile,wide", [
    (4096, 512, 64, 0),      # 0.5
    (4096, 576, 64, 1),      # 0.56
    (4096, 1024, 64, 1),     # 1
    (14336, 300, 64, 0),     # 1.09: 80.4 us wide, 71.0 narrow
    (4096, 2500, 128, 0),    # 1.25: 140 / 118
    (32000, 300, 128, 1),    # 1.46: 104 / 123
    (4096, 1500, 64, 1),     # 1.5
    (4096, 4096, 128, 1),    # 2
    (32000, 4096, 128, 1),   # 15.6
    (4224, 1024, 64, 0),     # not a multiple of 256 rows
])
def test_dense_products(gemm_wide, n, m, tile, wide):
    assert gemm_wide(0, n, m, 1, tile) == wide


# Mixtral shape (eight experts, top-2), tokens and slots per tile: the up projection (w1 and w3), the down projection
@pytest.mark.parametrize("tokens,tile,up,down", [
    (137, 64, 0, 0), (200, 64, 0, 0), (257, 64, 0, 1), (301, 128, 1, 0), (400, 128, 1, 0), (450, 128, 1, 0), (500, 128, 1, 1), (600, 128, 1, 1),
    (873, 128, 1, 1), (1000, 128, 0, 0), (1500, 128, 1, 1), (2048, 128, 1, 0), (4096, 128, 1, 0),
])
def test_routed_layers(gemm_wide, tokens, tile, up, down):
    assert gemm_wide(1, 2 * 14336, 2 * tokens, 8, tile) == up
    assert gemm_wide(0, 4096, 2 * tokens, 8, tile) == down


def test_a_wide_launch_is_at_least_half_a_round_and_its_last_round_more_than_a_third(gemm_wide):
    for n in (256, 1024, 4096, 5120, 14336, 32000):
        for m in range(96, 4097, 61):
            for tile in (64, 128):
                grid = n // 256 * -(-m // tile)
                if gemm_wide(0, n, m, 1, tile):
                    assert grid > 128 and (grid >= 2560 or grid % 256 == 0 or grid % 256 > 85), (n, m, tile)
