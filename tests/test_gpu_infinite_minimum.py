"""Blocks whose minimum is infinite (the f16 `m` of Q4_1 and Q5_1: an overflow in a converter), in the last block of a row and over
numbers of K steps that do and do not fill a round of the kernels' request rings: the streaming products give the infinities
`vec_dot_unopt` gives (candle-core/src/quantized/k_quants.rs), and no step beyond the end of K turns them into NaN."""
import numpy as np
import pytest

import candle_amd
import pyoracle as O
from helpers import activations, make_weights, rms

pytestmark = pytest.mark.gpu

BLOCK = {O.Q4_1: 20, O.Q5_1: 24}


def with_infinite_minimum(dt, w, rows, cols, at, sign=1):
    """The blocks of a [rows, cols] matrix with the last minimum of row `at` replaced."""
    b = np.array(w, copy=True).view(np.uint8).reshape(rows, cols // 32, BLOCK[dt])
    b[at, -1, 2:4] = np.array([sign * np.inf], dtype=np.float16).view(np.uint8)
    return b.reshape(-1)


# 25664 rows of n: the kernels whose waves walk all of K, two requests ahead and, from 24 steps of 128 on, six; 272: the one whose
# waves share K.  3, 4 and 25 steps.
@pytest.mark.parametrize("dt", [O.Q4_1, O.Q5_1])
@pytest.mark.parametrize("n,k", [(272, 384), (25664, 384), (25664, 512), (25664, 3200)])
def test_dense_products(dt, n, k):
    w = with_infinite_minimum(dt, O.fill_normal_quantized(n + k + dt, dt, n, k, 0.02), n, k, at=17)
    w = with_infinite_minimum(dt, w, n, k, at=18, sign=-1)
    lin = candle_amd.QMatMul(dt, w, n, k)
    x = activations(9, k, seed=k)
    got, want = lin.forward(x), O.matmul(dt, x, w, n)
    assert np.isinf(want[:, 17:19]).all() and np.isfinite(np.delete(want, (17, 18), axis=1)).all()
    assert np.array_equal(got, want)
    lin.close()


# The infinity in w3 of expert 0: its intermediate holds one, the block's scale is infinite and every output of its tokens NaN.
@pytest.mark.parametrize("dt", [O.Q4_1, O.Q5_1])
@pytest.mark.parametrize("H", [384, 512])
def test_layers(dt, H):
    F, E, k, T = 256, 4, 2, 6
    w1, w3, w2, _ = make_weights(H, F, E, dt, seed=3)
    w3[0] = with_infinite_minimum(dt, w3[0], F, H, at=40)
    gate = O.fill_normal(77, E * H, 0.0, 0.02).reshape(E, H)
    ref = O.Layer(H, F, E, k, dt, gate, w1, w3, w2)
    gpu = candle_amd.SparseMoeBlock(H, F, E, k, dt, gate, w1, w3, w2)
    xs = activations(T, H, seed=8)
    got = gpu.forward(xs)
    want = ref.forward(xs, logits=gpu.last_logits(T))
    lost = np.isnan(want).all(axis=1)
    assert lost.any() and not lost.all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    # (two weighted outputs per token are added, each exact: a few last places at most)
    assert np.abs(got[~lost] - want[~lost]).max() <= 1e-6 * rms(want[~lost])
    gpu.close()
