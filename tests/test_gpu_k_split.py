"""Tiled K-quant products whose workgroups share K between their waves (two or four parts), against the oracle's
`k_quants::matmul` (candle-core/src/quantized/k_quants.rs:1873-1920): numbers of super-blocks that do and do not divide by the
parts, last tiles that end in every kind of operand, and whole layers whose down projection is split."""
import os

import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, make_pair, rms

pytestmark = pytest.mark.gpu

CORES = max(1, min(16, len(os.sched_getaffinity(0))))
TOL = 1e-4   # max-abs error relative to rms(output): f32 sums over super-blocks in another order (as in test_gpu_qlinear.py)


# the rows of each line take: 64 slots in four parts, 64 in two, 128 in two (Q5K takes one part for some of them); k = 4352 and
# 4608: 17 and 18 super-blocks
@pytest.mark.parametrize("dt", [O.Q2K, O.Q3K, O.Q4K, O.Q5K, O.Q6K])
@pytest.mark.parametrize("n,k,rows", [
    (4096, 4352, (161, 177, 192, 250, 256)),
    (4096, 4608, (304, 385, 449, 500, 512)),
    (4096, 4352, (641, 660, 700, 750, 777, 800)),
])
def test_dense_products(dt, n, k, rows):
    w = O.fill_normal_quantized(n + k + dt, dt, n, k, 0.02)
    lin = candle_amd.QMatMul(dt, w, n, k)
    x = activations(max(rows), k, seed=n + dt)
    want = O.matmul(dt, x, w, n, simd=True, threads=CORES)
    for m in rows:
        got = lin.forward(x[:m])
        assert np.abs(got - want[:m]).max() <= TOL * rms(want), m
    lin.close()


# Eight experts, top-2: the down projection (H rows over F) in four parts of 64 slots and in two of 128.  The bar is that of a
# narrow K-quant layer, 2e-3 and 2e-4 rms at F = 14336 and sqrt(14336 / F) times that (a last bit of an f32 sum moves a value of
# the intermediate by one quantisation step now and then); one row in twenty may hold a step beyond the first.
@pytest.mark.parametrize("dt,dt_down", [(O.Q4K, None), (O.Q4K, O.Q6K), (O.Q5K, None)])
@pytest.mark.parametrize("H,F,tokens", [(512, 4352, (150, 300)), (4096, 2816, (260,))])
def test_layers(dt, dt_down, H, F, tokens):
    ref, gpu = make_pair(H, F, 8, 2, dt, seed=31, dt_down=dt_down)
    widen = float(np.sqrt(14336.0 / F))
    for T in tokens:
        xs = activations(T, H, seed=T)
        got = gpu.forward(xs)
        want = ref.forward(xs, logits=gpu.last_logits(T), simd=True, threads=CORES)
        beyond = np.nonzero(np.abs(got - want).max(axis=1) > 2e-3 * widen * rms(want))[0]
        assert beyond.size <= T // 20, (T, beyond.size)
        assert rms(got - want) <= 2e-4 * widen * rms(want), T
    gpu.close()
