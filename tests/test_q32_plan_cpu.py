"""The lines that choose the kernels of the 32-element formats (csrc/q32_plan.hpp), on the host: what they say beside the sizes they were measured at."""
import pytest

import plan_lib


@pytest.fixture(scope="module")
def plan():
    lib = plan_lib.load()
    if lib is None:
        pytest.skip("needs g++")
    return lib


# (H, F, lists, top-k, direct, always on, tokens) -> 1: fine up projection, + 2: fine down projection.  us, coarse / fine
@pytest.mark.parametrize("args,want", [
    ((1024, 3584, 8, 2, 1, 0, 16), 3),       # 37.3 / 26.8
    ((1024, 3584, 8, 2, 1, 0, 40), 3),
    ((1024, 3584, 8, 2, 1, 0, 65), 3),       # Q4_1, layer: 60.5 / 37.7
    ((1024, 3584, 8, 2, 1, 0, 94), 3),       # 71 / 46
    ((4096, 14336, 8, 2, 1, 0, 2), 3),       # up 85 / 56, 4 of 8 lists
    ((4096, 14336, 8, 2, 1, 0, 3), 3),       # Q5_1, layer: 200 / 131
    ((4096, 14336, 8, 2, 1, 0, 8), 0),       # 93 / 97
    ((2048, 1408, 48, 4, 1, 0, 33), 1),      # Q5_0, four layers: 388 / 362
    ((4096, 0, 1, 1, 0, 0, 16), 3),          # dense products: 21.4 / 11.4
    ((4096, 0, 1, 1, 0, 0, 96), 3),          # 28.4 / 25.4
    ((4096, 0, 1, 1, 0, 0, 112), 1),         # 28.4 / 27.7, 512: 28.9 / 30.8
    ((256, 512, 128, 1, 0, 0, 400), 0),      # layer 35.7 / 52.2
    ((256, 512, 128, 1, 0, 0, 640), 0),      # 40.8 / 67.1
    ((1024, 2816, 16, 1, 1, 0, 260), 0),     # 60.9 / 96.1
    ((4096, 5632, 1, 1, 0, 1, 113), 0),      # always on, beside 48 experts: 272 / 329
    ((2048, 5632, 1, 1, 0, 1, 16), 3),
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
