"""4^3 blocks, four samples to a wave (csrc/step_quads.hip) at the edges of what it works on, against the CPU oracle in
fp64: groups of samples and of blocks that are not full, the shortest and the longest history, batches in chunks."""

import pytest
import torch

from helpers import ATOL, RTOL, assert_close, make_acts, make_params
from test_routes import BLOCKS, QUADS, route

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# the rows' blocks in workgroups of four, three, two and one; one, two and more groups of samples, the last one of
# every size; two to nine iterations.  The forward is this file's with more than six pairs of block and sample to a CU, the
# backward where the last column says so: a walk of 32 at least, groups that are nearly full, more than half of the places of
# its waves taken
@pytest.mark.parametrize("shape,batch,inner,quads", [
    ((4, 4, 4), 4, 2, False), ((4, 8, 12), 5, 3, False), ((8, 8, 20), 7, 2, False), ((8, 4, 36), 6, 9, False),
    ((32, 32, 4), 25, 3, False), ((32, 32, 8), 14, 2, False), ((32, 32, 12), 11, 9, False), ((32, 32, 20), 5, 2, False),
    ((20, 28, 28), 7, 3, False),
    ((32, 32, 32), 16, 8, True), ((32, 32, 32), 31, 7, True), ((16, 16, 16), 256, 4, True), ((32, 32, 36), 32, 2, True),
    ((40, 44, 44), 16, 2, True), ((40, 44, 44), 4, 8, True), ((40, 44, 44), 16, 9, False), ((48, 48, 60), 16, 2, True)], ids=str)
@pytest.mark.parametrize("residual", [False, True], ids=["chain", "residual"])
@pytest.mark.parametrize("activation", ["silu", "tanh"])
def test_chain_against_the_oracle(shape, batch, inner, quads, residual, activation):
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    print(f"quads, chain {shape} B={batch} inner={inner} residual={residual} {activation} backward here: {quads}", flush=True)
    pairs = batch * shape[0] * shape[1] * shape[2] // 64
    assert (route(shape, batch, inner, 4, residual) == QUADS) == (pairs > 6 * 256)
    assert (route(shape, batch, inner, 4, residual, backward=1) == QUADS) == quads
    g = torch.Generator().manual_seed(3)
    w, b, r = make_params(shape, seed=11)
    if inner >= 7:
        w, r = w * 0.5, r * 0.5
    params = [w, b, r, *((a + 0.2 * torch.randn(shape, generator=g)) for a in (1, 0))]
    x, gy = (make_acts(batch, shape, seed=s) for s in (12, 13))
    run = BodyRunner(*(t.to(DEV) for t in params), batch, inner, 2, 4, activation, fused=True, outer_residual=residual)
    got = [run.forward(x.to(DEV)).clone(), *(t.clone() for t in run.backward(gy.to(DEV)))]
    for name, a, e in zip("y dweight dbias dscale dgamma dbeta dx".split(), [run.forward(x.to(DEV)), *run.backward(gy.to(DEV))], got):
        assert torch.equal(a, e), f"{name}: two runs differ"
    want = network_forward_backward([t.double() for t in params], x.double(), gy.double(), inner_iterations=inner,
                                    outer_iterations=2, block_size=4, activation=activation, outer_residual=residual)
    for name, a, e in zip("y dweight dbias dscale dgamma dbeta dx".split(), got, want):
        # an entry of the gradients is a sum over the batch, and its error goes with its terms (2e-7 of the array's rms)
        assert_close(a, e, RTOL, ATOL * max(1.0, e.pow(2).mean().sqrt().item()), name)


@pytest.mark.parametrize("room,want", [(4, QUADS), (3, QUADS), (2, BLOCKS), (0, BLOCKS)], ids=str)
def test_backward_with_room_for_fewer_chunks(room, want):
    """A batch in four chunks with room for the gradients of three: three longer ones.  Two would fill half of the places only, and the
    step goes to the general kernels."""
    from gridnet_amd import native as n
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    shape, batch, inner = (32, 32, 32), 64, 4
    nbytes = n.lib.gridnet_hip_fused_workspace_bytes(batch, *shape, inner, 4, 1) - (4 - room) * 31 * 32 ** 3 * 4
    print(f"quads, backward {shape} B={batch} inner={inner}, room for {room} chunks", flush=True)
    assert route(shape, batch, inner, 4, backward=1, workspace=nbytes) == want
    g = torch.Generator().manual_seed(3)
    params = [*make_params(shape, seed=11), *((a + 0.2 * torch.randn(shape, generator=g)) for a in (1, 0))]
    x, gy = (make_acts(batch, shape, seed=s) for s in (12, 13))
    run = BodyRunner(*(t.to(DEV) for t in params), batch, inner, 1, 4, "silu", fused=True)
    run.fb_ws_bytes, run.fb_ws = nbytes, torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    run.forward(x.to(DEV))
    got = run.backward(gy.to(DEV))
    want = network_forward_backward([t.double() for t in params], x.double(), gy.double(), inner_iterations=inner,
                                    outer_iterations=1, block_size=4, activation="silu")[1:]
    for name, a, e in zip("dweight dbias dscale dgamma dbeta dx".split(), got, want):
        assert_close(a, e, RTOL, ATOL * max(1.0, e.pow(2).mean().sqrt().item()), name)


def test_an_infinite_gradient_stays_within_the_taps_reach():
    """The last step of the residual loop has no LayerNorm behind it that would spread a non-finite gradient over its sample."""
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    shape, batch, inner, at = (32, 32, 36), 32, 2, (9, 13, 16)  # the first cell of a row of its block
    print(f"quads, residual {shape} B={batch} inner={inner}, an infinite gradient", flush=True)
    g = torch.Generator().manual_seed(3)
    params = [*make_params(shape, seed=11), *((a + 0.2 * torch.randn(shape, generator=g)) for a in (1, 0))]
    x, gy = (make_acts(batch, shape, seed=s) for s in (12, 13))
    run = BodyRunner(*(t.to(DEV) for t in params), batch, inner, 1, 4, "tanh", fused=True, outer_residual=True)
    assert route(shape, batch, inner, 4, 1, backward=1) == QUADS and route(shape, batch, inner, 4, 2, backward=1) == BLOCKS
    run.forward(x.to(DEV))
    bad = gy.clone()
    bad[5][at] = float("inf")
    got = [t.clone().cpu() for t in run.backward(bad.to(DEV))]
    want = network_forward_backward([t.double() for t in params], x.double(), gy.double(), inner_iterations=inner,
                                    outer_iterations=1, block_size=4, activation="tanh", outer_residual=True)[1:]
    away = torch.stack(torch.meshgrid(*(torch.arange(n) for n in shape), indexing="ij")).sub(torch.tensor(at).view(3, 1, 1, 1))
    away = away.abs().amax(0)
    # an iteration of the reverse sweep carries it one cell further, the first one none; gradients of weights are worked
    # out where the weight's tap reads from
    for name, a, e, reach in zip("dweight dbias dscale dgamma dbeta".split(), got, want, (2, 1, 1, 2, 2)):
        a, e = a[..., away > reach], e[..., away > reach]
        assert_close(a, e, RTOL, ATOL * max(1.0, e.pow(2).mean().sqrt().item()), name)
    others = [s for s in range(batch) if s != 5]
    assert_close(got[5][others], want[5][others], what="dx")
