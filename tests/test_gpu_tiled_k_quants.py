"""The tiled K-quant product at the edges of its tiles, against the oracle's `k_quants::matmul`
(candle-core/src/quantized/k_quants.rs:1873-1920): tiles of 64 and 128 rows, workgroups of eight waves (n a multiple of
256) and of four, and row counts that leave the last tile with every number of live 16-row operands the K loop exists
for; the streaming kernels with two row tiles per pass around their own edges; the pass that quantises rows."""
import os

import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, rms

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
# next super-block is multiplied.  n = 24576 gives eight-wave workgroups with two weight operands per wave where Q4K and Q2K
# are concerned, 12416 four-wave ones; Q3K, Q5K and Q6K take one operand per wave in both.  Last tiles of 1, 2, 3, 4 operands.
@pytest.mark.parametrize("dt", K_QUANTS)
@pytest.mark.parametrize("n,k", [(24576, 768), (12416, 1024)])
def test_every_number_of_live_operands_in_tiles_of_64_rows(dt, n, k):
    check(dt, n, k, (96, 111, 128, 130, 150, 176, 192), simd=True)


@pytest.mark.parametrize("n", [272, 8192])   # 16-row and 64-row workgroups
def test_two_row_tiles_per_pass_of_q6k(n):
    check(O.Q6K, n, 768, (16, 17, 31, 32, 33, 49, 64, 65))


@pytest.mark.parametrize("rows,k", [(1, 256), (3, 768), (256, 4096), (257, 4096 - 256), (1023, 4096), (1025, 4096), (331, 14336)])
def test_rows_quantised_with_one_two_and_four_blocks_per_wave(rows, k):
    # 4096 and 16384 blocks are where a wave takes two and four of them; odd counts leave the last wave's places empty
    x = activations(rows, k, seed=rows + k)
    x[rows // 2, :256] = 0.0
    assert np.array_equal(candle_amd.quantize_act(O.Q8K, x), O.quantize(O.Q8K, x))
