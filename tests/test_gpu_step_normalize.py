"""The backward with per-window normalisation where its sums could lose digits (csrc/step_fast.hip: they are formed from the
deltas and the pre-activations without their bias): biases far above the rest of the pre-activation, inputs far from zero,
against the CPU oracle in fp64."""

import pytest
import torch

from helpers import ATOL, RTOL, assert_close, make_acts, make_params
from test_gpu_step import oracle, run_op

pytestmark = pytest.mark.gpu


# one and two cells per thread, several slots to a workgroup; a slot of eight waves, of four, of one, half a wave
@pytest.mark.parametrize("shape,batch,inner,bs", [((8, 8, 8), 2, 5, 8), ((40, 48, 56), 5, 3, 8), ((16, 16, 16), 3, 4, 4),
                                                  ((32, 32, 32), 40, 3, 4)], ids=str)
@pytest.mark.parametrize("bias,offset", [(0.0, 0.0), (100.0, 0.0), (0.0, 100.0)], ids=["plain", "bias", "offset"])
def test_gradients_with_large_bias_or_offset(shape, batch, inner, bs, bias, offset):
    w, b, r = make_params(shape, seed=11)
    b = b + bias * torch.sign(b)
    x, gy = make_acts(batch, shape, seed=12) + offset, make_acts(batch, shape, seed=13)
    # a linear activation where the bias decides its side: every cell keeps clear of the kink by the bias
    activation = "leaky_relu" if bias else "silu"
    y, grads = run_op(w, b, r, x, gy, inner, bs, 1e-5, True, activation)
    ey, egrads = oracle(w, b, r, x, gy, inner, bs, 1e-5, True, activation)
    # values of the size of bias and offset are rounded at that size, a few ulp (6e-8) per iteration
    assert_close(y, ey, RTOL, ATOL * max(1.0, (bias + offset) / 10), "y")
    for name, g, e in zip(("dweight", "dbias", "dscale", "dx"), grads, egrads):
        # an entry is a sum over the batch and the iterations, and its error goes with its terms (2e-7 of the array's rms)
        assert_close(g, e, RTOL, ATOL * max(1.0, e.pow(2).mean().sqrt().item()), name)
