"""The costs that choose a tiled K-quant product's slot tile and the parts its workgroups cut K into, as a program on the host:
the choices beside their lines, that every choice is one the kernels exist for, over sizes of all orders, and what the sizes of the
GPU tests reach."""
import pytest

import plan_lib

Q2K, Q3K, Q4K, Q5K, Q6K = 10, 11, 12, 13, 14


class Plan:
    """Choices as 1000 * tile + parts; a streamed product 0, a streamed down projection 1000 * tile of the up projection."""

    def __init__(self, lib):
        self.lib = lib

    def dense(self, dt, n, k, m):
        c = self.lib.dense_kernel(dt, n, k, m)
        return c // 1000 * 1000 + c % 1000 // 10

    def layer(self, dt, H, F, tokens, top_k, E, dt_down=None):
        args = (dt, dt_down or dt, H, F, tokens, top_k, E)
        up, down = self.lib.up_kernel(*args), self.lib.down_kernel(*args)
        assert up % 1000 // 10 == 1 and (not down or down // 1000 == up // 1000)
        return up // 1000 * 1000 + down % 1000 // 10


@pytest.fixture(scope="module")
def plan():
    lib = plan_lib.load()
    if lib is None:
        pytest.skip("needs g++")
    return Plan(lib)


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
    (Q4K, 4096, 14336, 148, 64002), (Q5K, 4096, 14336, 154, 64002),                                      # 273 / 260, 385 / 335; 128 slots 271, 343
    (Q4K, 4096, 14336, 240, 128002), (Q4K, 4096, 14336, 301, 128002),                                    # 395 / 323, 371 / 354
    (Q4K, 4096, 14336, 640, 128001), (Q4K, 4096, 14336, 3000, 128001),                                   # two parts 715 / 695, 2480 / 2507
    (Q6K, 4096, 14336, 200, 128002), (Q5K, 4096, 14336, 260, 128002), (Q5K, 4096, 14336, 777, 128001),   # 395 / 325, 547 / 408; 1021 / 903
    (Q6K, 1024, 3584, 137, 64000), (Q4K, 1024, 3584, 260, 128000),                                        # 50, four parts 52; 66 / 55, four parts 57
    (Q4K, 1024, 3584, 160, 64004), (Q4K, 1024, 3584, 517, 64002), (Q4K, 1024, 3584, 1000, 128002),       # 49 / 46, 100 / 79, 126 / 115
])
def test_routed_layers(plan, f, H, F, tokens, want):
    assert plan.layer(f, H, F, tokens, 2, 8) == want


# Few super-blocks of w2, long lists: a streaming pass costs little less than with many.  us per step, tiled / streamed
@pytest.mark.parametrize("dt,H,F,tokens,top_k,E", [
    (Q4K, 3840, 256, 3089, 2, 34),    # 195 / 511
    (Q4K, 3840, 256, 1160, 2, 34),    # 128 / 251
    (Q4K, 768, 256, 3586, 1, 42),     # 67 / 138
    (Q4K, 768, 256, 664, 6, 41),      # 65 / 88
    (Q5K, 256, 256, 5337, 1, 66),     # 66 / 103
    (Q3K, 3328, 256, 1307, 2, 21),    # 112 / 179
    (Q6K, 256, 512, 2699, 2, 80),     # 69 / 113
    (Q4K, 256, 7168, 4857, 1, 16),    # Zipf loads: 199 / 331
])
def test_tiled_down_projections_of_long_lists(plan, dt, H, F, tokens, top_k, E):
    assert plan.layer(dt, H, F, tokens, top_k, E) % 1000 > 0


def test_few_super_blocks_of_a_dense_product(plan):
    assert plan.dense(Q4K, 4096, 512, 440)      # 10.7 to 11.3, streamed 18.3
    assert plan.dense(Q5K, 4096, 768, 332)      # 13.7, 17.3
    assert plan.dense(Q4K, 1152, 1280, 1530)    # 22.8, 27.6
    assert not plan.dense(Q2K, 1024, 14336, 480)   # 49; four parts 61
    assert plan.dense(Q4K, 4096, 4096, 2059) // 1000 == 128   # 92; 64 slots 104


def test_every_choice_has_a_kernel(plan):
    for f in (Q2K, Q3K, Q4K, Q5K, Q6K):
        for n in (128, 256, 384, 512, 1152, 4096, 14336, 65536):
            for k in (256, 512, 768, 1280, 4096, 14336):
                for m in (1, 95, 96, 113, 128, 129, 300, 777, 2049, 60000):
                    assert plan.dense(f, n, k, m) in (0, 64001, 64002, 64004, 128001, 128002), (f, n, k, m)
        for H, F in ((128, 256), (768, 512), (1024, 3584), (4096, 14336)):
            for E in (1, 2, 8, 60, 256):
                for per in (35, 64, 100, 129, 1000):
                    assert plan.layer(f, H, F, per * E, 1, E) in (64000, 64001, 64002, 64004, 128000, 128001, 128002), (f, H, F, E, per)


# What the GPU tests' sizes reach (eight experts, top-2): a change of the costs that empties one of them shows here.
def test_sizes_of_the_gpu_tests(plan):
    def layers(dt, H, F, tokens, dt_down=None):
        return {plan.layer(dt, H, F, T, 2, 8, dt_down) for T in tokens}

    # test_gpu_tiled_k_quants.py, test_layers: every format in tiles of 64 slots and of 128, tiled down projections of one to four parts
    for dt, dt_down in ((Q2K, None), (Q3K, None), (Q4K, None), (Q4K, Q6K), (Q5K, None), (Q6K, None)):
        assert layers(dt, 768, 512, (300, 360, 430, 600), dt_down) == {64001}
        assert 128002 in layers(dt, 768, 2048, (600, 660, 740), dt_down)
        assert layers(dt, 4096, 768, (270, 600), dt_down) == {64001, 128001}
        assert 64004 in layers(dt, 768, 1024, (200, 240, 270), dt_down) or dt == Q3K
    # test_gpu_parity.py
    for dt, dt_down in ((Q6K, None), (Q4K, Q6K), (Q6K, Q4K), (Q5K, None), (Q5K, Q6K), (Q2K, None), (Q2K, Q4K), (Q3K, None), (Q3K, Q5K)):
        assert layers(dt, 512, 1024, (500,), dt_down) == {64004}
    assert layers(Q4K, 512, 1024, (140, 150, 160, 200, 250, 270, 300, 400, 600)) == {64004}
    # test_gpu_k_split.py
    for dt in (Q2K, Q3K, Q4K, Q5K, Q6K):
        assert {plan.dense(dt, 4096, 4352, m) for m in (250, 256)} == {64004}
        assert {plan.dense(dt, 4096, 4608, m) for m in (304, 385, 449, 500, 512)} == {64002}
        assert {plan.dense(dt, 4096, 4352, m) for m in (641, 660, 700, 750, 777, 800)} == {128002 if dt in (Q3K, Q6K) else 64001}
        assert layers(dt, 4096, 2816, (260,)) == {128002}
    assert layers(Q4K, 512, 4352, (300,)) == {64004}
