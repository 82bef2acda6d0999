"""The tiled K-quant product at the edges of its tiles, against the oracle's `k_quants::matmul`
(candle-core/src/quantized/k_quants.rs:1873-1920): tiles of 64 and 128 rows, workgroups of eight waves (n a multiple of
256) and of four, and row counts that leave the last tile with every number of live 16-row operands the K loop exists
for; the streaming kernels with two row tiles per pass around their own edges; the pass that quantises rows."""
import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, rms

pytestmark = pytest.mark.gpu

TOL = 1e-4   # max-abs error relative to rms(output): f32 sums over super-blocks in another order (as in test_gpu_qlinear.py)
K_QUANTS = [O.Q2K, O.Q3K, O.Q4K, O.Q5K, O.Q6K]


def check(dt, n, k, rows):
    w = O.fill_normal_quantized(n + k + dt, dt, n, k, 0.02)
    lin = candle_amd.QMatMul(dt, w, n, k)
    x = activations(max(rows), k, seed=n + dt)
    want = O.matmul(dt, x, w, n)
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


@pytest.mark.parametrize("n", [272, 8192])   # 16-row and 64-row workgroups
def test_two_row_tiles_per_pass_of_q6k(n):
    check(O.Q6K, n, 768, (16, 17, 31, 32, 33, 49, 64, 65))


@pytest.mark.parametrize("rows,k", [(1, 256), (3, 768), (256, 4096), (257, 4096 - 256), (1023, 4096), (1025, 4096), (331, 14336)])
def test_rows_quantised_with_one_two_and_four_blocks_per_wave(rows, k):
    # 4096 and 16384 blocks are where a wave takes two and four of them; odd counts leave the last wave's places empty
    x = activations(rows, k, seed=rows + k)
    x[rows // 2, :256] = 0.0
    assert np.array_equal(candle_amd.quantize_act(O.Q8K, x), O.quantize(O.Q8K, x))
