"""The 32-element formats' kernels for launches of few workgroups (32 rows of F, 16 rows of H, K shared by the waves): bit for bit
the reference's scalar products (`vec_dot_unopt`, candle-core/src/quantized/k_quants.rs), at numbers of K steps that do and do not
fill a round of four, row counts around a pass of 16, and whole layers with idle experts, a row of workgroups per assignment and
lists of more than one pass."""
import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, make_pair, rms

pytestmark = pytest.mark.gpu

FORMATS = [O.Q4_0, O.Q4_1, O.Q5_0, O.Q5_1, O.Q8_0]


# 1, 4, 5 and 9 steps of 128; one row tile and an odd number of them; rows beside 16 and 32 (up to four rows take another kernel)
@pytest.mark.parametrize("dt", FORMATS)
@pytest.mark.parametrize("n,k", [(16, 128), (48, 512), (80, 640), (272, 1152)])
def test_dense_products_carry_the_reference_bits(dt, n, k):
    w = O.fill_normal_quantized(n + k + dt, dt, n, k, 0.02)
    lin = candle_amd.QMatMul(dt, w, n, k)
    x = activations(33, k, seed=n + dt)
    x[5, :32] = 0.0
    want = O.matmul(dt, x, w, n)
    for m in (5, 15, 16, 17, 32, 33):
        assert np.array_equal(lin.forward(x[:m]), want[:m]), m
    lin.close()


# 60 experts: a row of workgroups per assignment (3 tokens of top-4) and per expert (20); 4 experts: lists of two and three passes; F
# of a number of 32-row blocks that is no multiple of four
@pytest.mark.parametrize("dt", [O.Q4_0, O.Q5_1, O.Q8_0])
@pytest.mark.parametrize("H,F,E,k,tokens", [(256, 640, 60, 4, (1, 3, 20)), (384, 1152, 4, 2, (1, 8, 33, 70))])
def test_layers_carry_the_reference_bits(dt, H, F, E, k, tokens):
    ref, gpu = make_pair(H, F, E, k, dt, seed=5)
    for T in tokens:
        xs = activations(T, H, seed=T)
        got = gpu.forward(xs)
        want = ref.forward(xs, logits=gpu.last_logits(T))
        # (two to four weighted outputs per token are added, each exact: a few last places at most)
        assert np.abs(got - want).max() <= 1e-6 * rms(want), (T, np.abs(got - want).max() / rms(want))
    gpu.close()
