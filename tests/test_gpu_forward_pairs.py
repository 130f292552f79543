"""The chain's forward with 8^3 blocks (csrc/step_fast.hip) on both sides of the rule that takes two
elements per pass: odd batches, walks of even and odd length, an odd and an even number of iterations,
grids that are no cubes, against the CPU oracle in fp64."""

import pytest
import torch

from helpers import make_acts, make_params
from test_routes import BLOCKS, PAIRS, route

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shape,batch,inner,pairs", [
    ((40, 40, 40), 63, 2, True), ((40, 40, 40), 64, 3, True), ((40, 40, 40), 65, 2, False),
    ((48, 32, 40), 71, 3, False), ((64, 40, 48), 17, 2, True), ((16, 24, 8), 5, 2, True)], ids=str)
def test_against_oracle(shape, batch, inner, pairs):
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward

    print(f"forward {shape} B={batch} inner={inner}", flush=True)
    assert route(shape, batch, inner, 8) == (PAIRS if pairs else BLOCKS)
    g = torch.Generator().manual_seed(3)
    params = [*make_params(shape, seed=1), 1 + 0.2 * torch.randn(shape, generator=g), 0.2 * torch.randn(shape, generator=g)]
    x = make_acts(batch, shape, seed=2)
    run = BodyRunner(*(t.to(DEV) for t in params), batch, inner, 2, 8, "silu", fused=True, backward=False, forward_all=False)
    got = run.forward(x.to(DEV)).cpu().double()
    want = network_forward(*(t.double() for t in params), x.double(), inner_iterations=inner, outer_iterations=2,
                           block_size=8, activation="silu")
    # a cell is 2 * inner sums of 27 products and two LayerNorms of it: some 60 roundings of 6e-8 each per sum, of
    # values up to about ten
    assert (got - want).abs().max() <= 2 * inner * 60 * 6e-8 * 10
