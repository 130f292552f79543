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


# slots of eight waves, of four, of half a wave; 4^3 blocks see their neighbours' cells in the window
@pytest.mark.parametrize("shape,batch,bs", [((8, 8, 8), 1, 8), ((8, 8, 8), 800, 8), ((8, 8, 8), 3, 4), ((16, 8, 8), 1600, 4)], ids=str)
def test_the_derivative_is_that_of_the_side_the_forward_took(shape, batch, bs):
    """A bias that cancels the rest of the pre-activation to its last bit leaves the rounding error of that rest, which a fused
    multiply-add sees and a sum of the two does not: value and derivative have to come from the same number.  One tap of weight 1
    on whole numbers, so that all sums are exact and the CPU knows every intermediate value."""
    import numpy as np

    f32 = np.float32
    rng = np.random.default_rng(3)
    x = rng.integers(-60, 61, shape).astype(f32)
    eps, bias = f32(1e-5), np.zeros(shape, f32)
    padded = np.pad(x, 1)
    for p in range(0, shape[0], bs):
        for q in range(0, shape[1], bs):
            for r in range(0, shape[2], bs):
                win = padded[p:p + bs + 2, q:q + bs + 2, r:r + bs + 2] - x[p, q, r]  # kept less the block's first cell
                count = f32(1) / f32(win.size)
                mean = f32(win.sum(dtype=np.float64)) * count
                square = f32((win.astype(np.float64) ** 2).sum()) * count
                var = f32(np.float64(square) - np.float64(mean) * np.float64(mean))
                inv = f32(1) / (np.sqrt(var) + eps)
                bias[p:p + bs, q:q + bs, r:r + bs] = -(inv * (win[1:-1, 1:-1, 1:-1] - mean))
    w = torch.zeros(27, *shape)
    w[13] = 1
    scale = torch.full(shape, 2.0 ** 30)
    xs = torch.from_numpy(x).expand(batch, *shape).contiguous()
    y, (_, db, dr, _) = run_op(w, torch.from_numpy(bias), scale, xs, torch.ones_like(xs), 1, bs, float(eps), True, "relu")
    y, db, dr = y.cpu(), db.cpu(), dr.cpu()
    positive = y[0] > xs[0]
    assert 0.2 < positive.float().mean() < 0.8  # about half of the errors are
    assert torch.equal(db > 0, positive) and torch.equal(dr > 0, positive)
