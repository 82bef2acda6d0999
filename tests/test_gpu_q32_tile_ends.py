"""The tiled up projection of the 32-element formats, whose silu and re-quantisation follow the length of a tile: lists of many
lengths, whole tiles with a few slots in a second one among them, and an always-on expert whose last tile ends in each kind of
operand, bit for bit the reference's scalar products (`vec_dot_unopt`, candle-core/src/quantized/k_quants.rs)."""
import numpy as np
import pytest

import pyoracle as O
from helpers import activations, make_pair, rms

pytestmark = pytest.mark.gpu


# 32 experts, top-4: about 13 (where the tiled kernels start), 21, 37 and 65 rows per expert, each list of another length
@pytest.mark.parametrize("dt", [O.Q4_0, O.Q5_1, O.Q8_0])
@pytest.mark.parametrize("H,F,Fs", [(256, 384, 0), (128, 256, 128)])
def test_layers_carry_the_reference_bits(dt, H, F, Fs):
    ref, gpu = make_pair(H, F, 32, 4, dt, seed=9, Fs=Fs)
    for T in (105, 170, 301, 517, 529, 572):
        xs = activations(T, H, seed=T)
        got = gpu.forward(xs)
        want = ref.forward(xs, logits=gpu.last_logits(T))
        # (four or five weighted outputs per token are added, each exact: a few last places at most)
        assert np.abs(got - want).max() <= 1e-6 * rms(want), (T, np.abs(got - want).max() / rms(want))
    gpu.close()
