"""The step's kernels for small grids (csrc/step_fast.hip: few_pairs and, for 4^3 blocks, few_for_slots and
launch_bwd_slots) and those that take over where a CU gets more (block, element) pairs, on both sides of the line, against
the CPU oracle in fp64."""

import pytest
import torch

from helpers import ATOL, RTOL, acts_clear_of_kink, assert_close, make_acts, make_params
from test_gpu_step import oracle, run_op

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (pairs on 256 CUs): one block; the forward's line at two pairs per CU, the backward's at three with normalize and four
# without (65 is not split evenly); blocks that have a neighbour on one side only; ten inner iterations (at twenty the
# gradients reach 3e3 and torch's own fp32 evaluation on the CPU lies 1.3 to 1.5 times outside the bar); 256 blocks,
# whose workgroups have the whole batch in the backward.  4^3 blocks (few_for_slots, launch_bwd_slots): one slot and four of
# one cell per thread, two, four and eight of two, full and with elements missing; two and three samples, each a wave's
# with a copy of the gradients of its own, and three that a wave walks
@pytest.mark.parametrize("shape,batch,inner,bs", [(*c, 8) for c in [
    ((8, 8, 8), 1, 1), ((8, 8, 8), 3, 4), ((16, 16, 16), 64, 2), ((16, 16, 16), 65, 2), ((24, 32, 40), 17, 2), ((24, 32, 40), 18, 2),
    ((16, 16, 32), 48, 2), ((16, 16, 32), 64, 2), ((16, 16, 32), 65, 2), ((16, 8, 24), 2, 10), ((32, 64, 64), 1, 2),
    ((32, 64, 64), 2, 2)]] + [(*c, 4) for c in [
    ((4, 4, 4), 1, 2), ((8, 4, 12), 3, 4), ((16, 16, 16), 2, 10), ((24, 24, 20), 2, 2), ((24, 24, 20), 3, 4), ((16, 16, 16), 4, 2), ((16, 16, 16), 32, 2), ((16, 16, 16), 64, 2), ((16, 16, 16), 65, 2),
    ((32, 32, 16), 3, 2), ((32, 32, 16), 9, 2), ((32, 32, 16), 31, 2), ((32, 32, 16), 32, 2), ((32, 32, 16), 37, 2), ((32, 36, 36), 4, 2),
    ((32, 36, 36), 5, 2), ((32, 36, 36), 18, 2), ((48, 48, 36), 4, 4), ((48, 48, 36), 5, 4)]], ids=str)
@pytest.mark.parametrize("normalize", [False, True], ids=["plain", "normalize"])
@pytest.mark.parametrize("activation", ["silu", "leaky_relu"])
def test_step_on_both_sides_of_the_line(shape, batch, inner, bs, normalize, activation):
    print(f"small grid {shape} bs={bs} B={batch} inner={inner} normalize={normalize} {activation}", flush=True)
    w, b, r = make_params(shape, seed=11)
    if inner >= 8:
        w, r = w * 0.5, r * 0.5
    x = acts_clear_of_kink(w, b, r, batch, shape, inner, bs, 1e-5, normalize, activation, seed=12)
    gy = make_acts(batch, shape, seed=13)
    y, grads = run_op(w, b, r, x, gy, inner, bs, 1e-5, normalize, activation)
    ey, egrads = oracle(w, b, r, x, gy, inner, bs, 1e-5, normalize, activation)
    assert_close(y, ey, RTOL, ATOL, "y")
    for name, g, e in zip(("dweight", "dbias", "dscale", "dx"), grads, egrads):
        # An entry is a sum of batch x inner products; its rounding error goes with the size of those, 2e-7 of the rms of the
        # array (fp32, any order), not with what is left of the sum: 50 of these where the rms is above one.
        assert_close(g, e, RTOL, ATOL * max(1.0, e.pow(2).mean().sqrt().item()), name)


# the backward of a chain at the last batch of the small kernels, and with one sample more
@pytest.mark.parametrize("more", [0, 1], ids=["last", "next"])
@pytest.mark.parametrize("shape,batch,inner,bs", [
    ((16, 16, 32), 64, 2, 8), ((32, 32, 32), 16, 3, 8), ((24, 32, 40), 17, 2, 8), ((16, 16, 16), 64, 2, 4), ((16, 16, 16), 2, 4, 4),
    ((32, 32, 32), 3, 2, 4), ((32, 32, 32), 31, 2, 4), ((32, 36, 36), 4, 2, 4), ((48, 48, 36), 4, 4, 4), ((64, 64, 64), 1, 2, 4)],
    ids=str)
@pytest.mark.parametrize("residual", [False, True], ids=["chain", "residual"])
def test_chain_on_both_sides_of_the_line(shape, batch, inner, bs, residual, more):
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    batch += more
    print(f"small grid, chain {shape} bs={bs} B={batch} inner={inner} residual={residual}", flush=True)
    g = torch.Generator().manual_seed(3)
    params = [*make_params(shape, seed=11), *((a + 0.2 * torch.randn(shape, generator=g)) for a in (1, 0))]
    x, gy = (make_acts(batch, shape, seed=s) for s in (12, 13))
    run = BodyRunner(*(t.to(DEV) for t in params), batch, inner, 2, bs, "silu", fused=True, outer_residual=residual)
    got = [run.forward(x.to(DEV)).clone(), *run.backward(gy.to(DEV))]
    want = network_forward_backward([t.double() for t in params], x.double(), gy.double(), inner_iterations=inner,
                                    outer_iterations=2, block_size=bs, activation="silu", outer_residual=residual)
    for name, a, e in zip(("y", "dweight", "dbias", "dscale", "dgamma", "dbeta", "dx"), got, want):
        # the bound of above: an entry of the gradients is a sum over the batch, and its error goes with its terms
        assert_close(a, e, RTOL, ATOL * max(1.0, e.pow(2).mean().sqrt().item()), name)
