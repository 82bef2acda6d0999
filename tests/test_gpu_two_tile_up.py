"""The two-tile Q4_K up projection whose activation rows are staged in LDS: lists that end inside the first and inside the second
slot tile of a pass and lists of two passes, one, two and three super-blocks, with and without a dispatch pass, against the
oracle."""
import os

import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, make_pair, rms

pytestmark = pytest.mark.gpu

CORES = max(1, min(16, len(os.sched_getaffinity(0))))


# The bar is that of a narrow K-quant layer: 2e-3 and 2e-4 rms at F = 14336 and sqrt(14336 / F) times that (a last bit of an f32
# sum moves a value of the intermediate by one quantisation step now and then); one row in twenty may hold a step beyond it.
@pytest.mark.parametrize("dt_down", [None, O.Q6K])
@pytest.mark.parametrize("H,F,E,tokens", [
    (256, 512, 4, (27, 40, 66)),     # 13.5, 20, 33 rows per expert
    (768, 256, 4, (30, 64)),
    (512, 1024, 32, (215, 500)),     # lists from the dispatch pass
])
def test_layers(dt_down, H, F, E, tokens):
    ref, gpu = make_pair(H, F, E, 2, O.Q4K, seed=41, dt_down=dt_down)
    widen = float(np.sqrt(14336.0 / F))
    for T in tokens:
        xs = activations(T, H, seed=T)
        got = gpu.forward(xs)
        want = ref.forward(xs, logits=gpu.last_logits(T), simd=True, threads=CORES)
        beyond = np.nonzero(np.abs(got - want).max(axis=1) > 2e-3 * widen * rms(want))[0]
        assert beyond.size <= max(1, T // 20), (T, beyond.size)
        assert rms(got - want) <= 2e-4 * widen * rms(want), T
    gpu.close()


# The kernel rounds where the one that carries four slot tiles in registers does, over the same sums in the same order: the same
# bits.  (Q6K w2: its down kernels carry two tiles at most, so both runs share theirs.)
@pytest.mark.parametrize("H,F,E,tokens", [
    (256, 512, 4, (3, 8, 27, 40, 66)),
    (768, 256, 4, (30, 64)),
    (1280, 1024, 8, (50, 101)),
    (512, 1024, 32, (215, 500)),
])
def test_same_bits_as_four_tiles_in_registers(H, F, E, tokens):
    _, gpu = make_pair(H, F, E, 2, O.Q4K, seed=43, dt_down=O.Q6K)
    try:
        for T in tokens:
            xs = activations(T, H, seed=T + 1)
            got = {}
            for tiles in (2, 4):
                candle_amd.set_switch("slot_tiles", tiles)
                got[tiles] = gpu.forward(xs)
            assert np.array_equal(got[2], got[4]), T
    finally:
        candle_amd.set_switch("slot_tiles", 0)
    gpu.close()
