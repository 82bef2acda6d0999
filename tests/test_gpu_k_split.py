"""Tiled K-quant products whose workgroups share K between their waves (two or four parts), against the oracle's
`k_quants::matmul` (candle-core/src/quantized/k_quants.rs:1873-1920): numbers of super-blocks that do and do not divide by the
parts, last tiles that end in every kind of operand, and whole layers whose down projection is split.  Which kernel a size takes by
itself is a matter of costs (tests/test_gemm_split_plan_cpu.py has the sizes used here); the tests that name a kernel set it by the
library's switches."""
import os

import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, make_pair, rms

pytestmark = pytest.mark.gpu

CORES = max(1, min(16, len(os.sched_getaffinity(0))))
TOL = 1e-4   # max-abs error relative to rms(output): f32 sums over super-blocks in another order (as in test_gpu_qlinear.py)


# As the costs have it.  The rows of each line take: 64 slots in four parts (Q3K, Q5K and Q6K streamed below 250 rows); 64 in two; 128
# in two (Q3K, Q6K) or 64 in one (Q2K, Q4K, Q5K).  k = 4352 and 4608: 17 and 18 super-blocks
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


K_QUANTS = [O.Q2K, O.Q3K, O.Q4K, O.Q5K, O.Q6K]
KERNELS = [(64, 1), (64, 2), (64, 4), (128, 1), (128, 2)]   # (slots per tile, parts of K)


class Forced:
    """The down projection and dense products by the kernel for (tile, parts); parts 0: streamed."""

    def __init__(self, tile, parts):
        self.to = {"tile_slots": tile, "tiled_down": int(parts > 0), "k_parts": parts}

    def __enter__(self):
        for name, value in self.to.items():
            candle_amd.set_switch(name, value)

    def __exit__(self, *exc):
        for name, value in {"tile_slots": 0, "tiled_down": -1, "k_parts": 0}.items():
            candle_amd.set_switch(name, value)


# Fewer super-blocks than parts (k = 256: parts without any), a part one longer than the next (768, 1280), even parts (2048); last
# tiles of 1 to 4 and 1 to 8 operands, full and not.
@pytest.mark.parametrize("dt", K_QUANTS)
@pytest.mark.parametrize("n,k", [(128, 256), (384, 768), (256, 1280), (128, 2048)])
def test_every_kernel(dt, n, k):
    w = O.fill_normal_quantized(n + k + dt, dt, n, k, 0.02)
    lin = candle_amd.QMatMul(dt, w, n, k)
    x = activations(250, k, seed=n + dt)
    want = O.matmul(dt, x, w, n)
    for tile, parts in KERNELS:
        rows = (1, 17, 48, 63, 64, 65, 96, 177) if tile == 64 else (5, 32, 33, 63, 70, 96, 100, 127, 128, 129, 150, 250)
        with Forced(tile, parts):
            for m in rows:
                got = lin.forward(x[:m])
                assert np.abs(got - want[:m]).max() <= TOL * rms(want[:m]), (tile, parts, m)
    lin.close()


# The same over expert lists: tiled and streamed down projections of the same intermediate (the up projection does not change)
# differ by the order of their f32 sums alone -- n super-blocks' results added with an error of n 2^-24 of their sum of magnitudes
# each, less than n^1.5 2^-24 rms for sums of either sign: 1e-5 rms covers n = 9 ten times over.
@pytest.mark.parametrize("dt,dt_down", [(O.Q2K, None), (O.Q3K, None), (O.Q4K, None), (O.Q4K, O.Q6K), (O.Q5K, None), (O.Q6K, O.Q2K)])
@pytest.mark.parametrize("H,F", [(256, 768), (512, 2304)])
def test_every_kernel_over_lists(dt, dt_down, H, F):
    _, gpu = make_pair(H, F, 8, 2, dt, seed=33, dt_down=dt_down)
    for T in (140, 230, 410):
        xs = activations(T, H, seed=T)
        base = {}
        for tile, parts in [(64, 0), (128, 0)] + KERNELS:
            with Forced(tile, parts):
                got = gpu.forward(xs)
            base.setdefault(tile, got)
            assert np.abs(got - base[tile]).max() <= 1e-5 * rms(got), (T, tile, parts)
    gpu.close()


# Eight experts, top-2.  As the costs have it, four parts of 64 slots (H = 512, 300 tokens: Q4K), two of 128 (H = 4096) or streamed
# (the others).  The bar is that of a
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
