"""The tiled K-quant product at the edges of its tiles, against the oracle's `k_quants::matmul`
(candle-core/src/quantized/k_quants.rs:1873-1920): tiles of 64 and 128 rows, workgroups of eight waves and of four, and row
counts that leave the last tile with every number of live 16-row operands the K loop exists for, over one super-block and
over three and four; whole layers, whose up projection is a kernel of its own; the streaming kernels with two row tiles per
pass around their own edges; the pass that quantises rows."""
import os

import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import FlipExplainer, activations, make_pair, rms

pytestmark = pytest.mark.gpu

TOL = 1e-4   # max-abs error relative to rms(output): f32 sums over super-blocks in another order (as in test_gpu_qlinear.py)
K_QUANTS = [O.Q2K, O.Q3K, O.Q4K, O.Q5K, O.Q6K]


CORES = max(1, min(16, len(os.sched_getaffinity(0))))


def check(dt, n, k, rows, simd=False):
    # simd: the oracle's AVX2 inner loops, which agree with its scalar ones to 1e-6 relative (quantized_tests.rs:869-876)
    w = O.fill_normal_quantized(n + k + dt, dt, n, k, 0.02)
    lin = candle_amd.QMatMul(dt, w, n, k)
    x = activations(max(rows), k, seed=n + dt)
    want = O.matmul(dt, x, w, n, simd=simd, threads=CORES if simd else 1)
    for m in rows:
        got = lin.forward(x[:m])
        assert np.abs(got - want[:m]).max() <= TOL * rms(want), m
    lin.close()


@pytest.mark.parametrize("dt", K_QUANTS)
@pytest.mark.parametrize("n", [24576, 12416])
def test_tiles_of_64_rows(dt, n):
    check(dt, n, 512, (96, 97, 112, 128, 129, 161, 177))


@pytest.mark.parametrize("dt", K_QUANTS)
@pytest.mark.parametrize("n", [65536, 65664])
def test_tiles_of_128_rows(dt, n):
    check(dt, n, 256, (96, 97, 113, 128, 129, 161, 193))


# An odd and an even number of super-blocks, three at least: both LDS buffers are filled again, and what was requested for the
# next super-block is multiplied.  n = 16640 gives eight-wave workgroups with two weight operands per wave where Q4K and Q2K
# are concerned, 12416 four-wave ones; Q3K, Q5K and Q6K take one operand per wave in both.  Last tiles of 1, 2, 3, 4 operands.
@pytest.mark.parametrize("dt", K_QUANTS)
@pytest.mark.parametrize("n,k", [(16640, 768), (12416, 1024)])
def test_every_number_of_live_operands_in_tiles_of_64_rows(dt, n, k):
    check(dt, n, k, (96, 111, 128, 130, 150, 176, 192), simd=True)


# the same of tiles of 128 rows: eight-wave workgroups (32768) and four-wave ones, last tiles of 1 to 8 operands
@pytest.mark.parametrize("dt", K_QUANTS)
@pytest.mark.parametrize("n,k", [(32768, 768), (32896, 1024)])
def test_every_number_of_live_operands_in_tiles_of_128_rows(dt, n, k):
    check(dt, n, k, (130, 150, 176, 192, 200, 220, 239, 256), simd=True)


# Layers of eight experts, top-2, whose lists end in different operands of a tile.  Up projection: tiles of 64 slots and of 128,
# four-wave workgroups (F = 512, 768) and eight-wave ones (F = 2048).  Down, as the costs have it (tests/test_gemm_split_plan_cpu.py):
# one part (F = 512, 768; eight waves at H = 4096), two parts of 128 slots (F = 2048), four of 64 (F = 1024; Q3K streamed).  Every down
# kernel at every size: test_gpu_k_split.py.
# The bar is that of any narrow K-quant layer: an f32 sum in another order moves a value of the intermediate by one quantisation
# step now and then, which weighs sqrt(14336 / F) times what it does at F = 14336 (there 2e-3 max and 2e-4 rms).  A row beyond
# it has to be within it once such steps, four at most, are taken out (FlipExplainer).
@pytest.mark.parametrize("dt,dt_down", [(O.Q2K, None), (O.Q3K, None), (O.Q4K, None), (O.Q4K, O.Q6K), (O.Q5K, None), (O.Q6K, None)])
@pytest.mark.parametrize("H,F,tokens", [(768, 1024, (200, 240, 270)), (768, 512, (300, 360, 430, 600)), (768, 2048, (600, 660, 740)), (4096, 768, (270, 600))])
def test_layers(dt, dt_down, H, F, tokens):
    ref, gpu = make_pair(H, F, 8, 2, dt, seed=21, dt_down=dt_down)
    widen = float(np.sqrt(14336.0 / F))
    for T in tokens:
        xs = activations(T, H, seed=T)
        got = gpu.forward(xs)
        want = ref.forward(xs, logits=gpu.last_logits(T), simd=True, threads=CORES)
        bar = 2e-3 * widen * rms(want)
        beyond = np.nonzero(np.abs(got - want).max(axis=1) > bar)[0]
        assert beyond.size <= T // 20, (T, beyond.size)
        idx, weights = gpu.last_routing(T)[:2]
        for t in beyond:
            left, found = FlipExplainer(ref).explain(got[t] - want[t], xs[t], idx[t], weights[t], bar)
            assert left <= bar, (T, t, left / rms(want), found)
        assert rms(got - want) <= 2e-4 * widen * rms(want), T
    gpu.close()


@pytest.mark.parametrize("n", [272, 8192])   # 16-row and 64-row workgroups
def test_two_row_tiles_per_pass_of_q6k(n):
    check(O.Q6K, n, 768, (16, 17, 31, 32, 33, 49, 64, 65))


@pytest.mark.parametrize("rows,k", [(1, 256), (3, 768), (256, 4096), (257, 4096 - 256), (1023, 4096), (1025, 4096), (331, 14336)])
def test_rows_quantised_with_one_two_and_four_blocks_per_wave(rows, k):
    # 4096 and 16384 blocks are where a wave takes two and four of them
    x = activations(rows, k, seed=rows + k)
    x[rows // 2, :256] = 0.0
    assert np.array_equal(candle_amd.quantize_act(O.Q8K, x), O.quantize(O.Q8K, x))


@pytest.mark.parametrize("blocks", [4095, 4096, 4097, 4111, 16383, 16384, 16385, 16386, 16387, 16399])
def test_rows_quantised_where_the_last_wave_has_places_left(blocks):
    # one block per wave below 4096 blocks, two from there (odd counts: one place empty), four from 16384 (one to three empty)
    x = activations(blocks, 256, seed=blocks)
    x[-1, 7] = 40.0
    assert np.array_equal(candle_amd.quantize_act(O.Q8K, x), O.quantize(O.Q8K, x))
