"""The lines that choose the kernels of the 32-element formats (csrc/q32_plan.hpp), on the host: what they say beside the sizes they were measured at."""
import pytest

import plan_lib


@pytest.fixture(scope="module")
def plan():
    lib = plan_lib.load()
    if lib is None:
        pytest.skip("needs g++")
    return lib


# (H, F, lists, top-k, direct, always on, slot tiles, tokens) -> 1: fine up projection, + 2: fine down projection.  us, coarse / fine
@pytest.mark.parametrize("args,want", [
    ((1024, 3584, 8, 2, 1, 0, 1, 16), 3),       # 37.3 / 26.8
    ((1024, 3584, 8, 2, 1, 0, 1, 40), 3),
    ((1024, 3584, 8, 2, 1, 0, 1, 64), 2),       # lists of a second pass: up 20.8 / 22.6
    ((4096, 14336, 8, 2, 1, 0, 1, 2), 3),       # up 85 / 56, 4 of 8 lists
    ((4096, 14336, 8, 2, 1, 0, 1, 8), 0),       # 93 / 97
    ((4096, 0, 1, 1, 0, 0, 1, 16), 3),          # dense products: 21.4 / 11.4
    ((4096, 0, 1, 1, 0, 0, 4, 96), 3),          # 28.4 / 25.4
    ((4096, 0, 1, 1, 0, 0, 4, 112), 1),         # 28.4 / 27.7, 512: 28.9 / 30.8
    ((2048, 2816, 8, 4, 1, 0, 1, 28), 1),       # down, empty workgroups counted: layer 53.6 / 60.3
    ((256, 512, 128, 1, 0, 0, 1, 400), 0),      # layer 35.7 / 52.2
    ((256, 512, 128, 1, 0, 0, 1, 640), 0),      # 40.8 / 67.1
    ((1024, 2816, 16, 1, 1, 0, 2, 260), 0),     # 60.9 / 96.1
    ((4096, 5632, 1, 1, 0, 1, 4, 89), 0),       # always on, beside 48 experts: 263 / 279
    ((4096, 5632, 1, 1, 0, 1, 4, 113), 0),      # 272 / 329
    ((2048, 5632, 1, 1, 0, 1, 1, 16), 3),
])
def test_fine_kernels(plan, args, want):
    assert plan.fine(*args) == want


# (tokens, top-k, experts), slots grouped by a dispatch pass.  us, streamed / tiled
@pytest.mark.parametrize("args,want", [
    ((120, 4, 60), 0),       # 8 rows per expert: 191 / 218
    ((170, 4, 60), 0),       # 11: 145 / 159
    ((220, 4, 60), 1),       # 15: 250 / 200
    ((320, 8, 214), 0),      # 12 rows, 20 passes: even over layers, 243 / 180 here
    ((1970, 1, 206), 1),     # 9.6 rows, 124 passes: 171 / 114
    ((1250, 1, 206), 1),     # 6.1 rows, 79 passes: means 1.05
    ((1200, 1, 206), 0),
    ((2772, 1, 248), 1),     # 667 / 377
    ((133, 6, 44), 1),       # 18 rows, 9 passes
    ((350, 2, 50), 1),       # 14 rows, 22 passes
    ((21, 64, 64), 1),       # above 20 rows
    ((150, 3, 32), 0),       # 14 rows, 10 passes
])
def test_tiled_kernels(plan, args, want):
    assert plan.tiled32(*args) == want
