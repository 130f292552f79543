"""Chains of steps with one inner iteration by whole rows (csrc/chain_rows.hip): plain, through the
runner, and gated, through the model's loop, against the CPU oracle in fp64.  Rows of every length covered,
tubes at all edges of the grid at once (4 x 4 rows), batches below and above what splits the batch over
workgroups, one outer step and several."""

import pytest
import torch

from helpers import assert_close, make_acts, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SHAPES = [((4, 4, 16), 4, 1, 1), ((4, 8, 32), 4, 5, 3), ((8, 16, 32), 8, 9, 2), ((8, 4, 16), 4, 40, 4),
          ((8, 8, 64), 8, 3, 3), ((16, 8, 64), 8, 1, 2)]
ids = ["x".join(map(str, s)) + f"-{b}-{o}" for s, _, b, o in SHAPES]


def inputs(shape, batch):
    g = torch.Generator().manual_seed(5)
    gamma, beta = 1 + 0.2 * torch.randn(shape, generator=g), 0.2 * torch.randn(shape, generator=g)
    return gamma, beta, make_acts(batch, shape, seed=6), make_acts(batch, shape, seed=7)


@pytest.mark.parametrize("activation", ["silu", "tanh"])
@pytest.mark.parametrize("shape,bs,batch,outer", SHAPES, ids=ids)
def test_plain_chain(shape, bs, batch, outer, activation):
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    print(f"rows chain {shape} B={batch} outer={outer} {activation}", flush=True)
    gamma, beta, x, gy = inputs(shape, batch)
    params = [*make_params(shape, seed=4), gamma, beta]
    run = BodyRunner(*(t.to(DEV) for t in params), batch, 1, outer, bs, activation, fused=True, forward_all=False)
    assert run.rows
    results = []
    for _ in range(2):
        results.append([run.forward(x.to(DEV)).clone(), *[t.clone() for t in run.backward(gy.to(DEV))]])
    alone = BodyRunner(*(t.to(DEV) for t in params), batch, 1, outer, bs, activation, fused=True, forward_all=False,
                       backward=False)
    assert torch.equal(alone.forward(x.to(DEV)), results[0][0])
    want = network_forward_backward([t.double() for t in params], x.double(), gy.double(), inner_iterations=1,
                                    outer_iterations=outer, block_size=bs, activation=activation)
    for name, a, b, e in zip(("y", "dweight", "dbias", "dscale", "dgamma", "dbeta", "dx0"), *results, want):
        assert torch.equal(a, b), name
        assert_close(a, e, rtol=2e-4, atol=2e-5, what=name)


@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
@pytest.mark.parametrize("batch", [2, 40])
def test_gradients_on_top_of_what_the_buffers_hold(batch, accumulate):
    from gridnet_amd import native as n
    from gridnet_amd.runner import BodyRunner

    shape, outer = (8, 8, 16), 3
    gamma, beta, x, gy = inputs(shape, batch)
    run = BodyRunner(*(t.to(DEV) for t in (*make_params(shape, seed=4), gamma, beta)), batch, 1, outer, 8, "silu",
                     fused=True)
    run.forward(x.to(DEV))
    want = [t.clone() for t in run.backward(gy.to(DEV))[:5]]
    old, n.OVERWRITE_PARAMS = n.OVERWRITE_PARAMS, 0 if accumulate else n.OVERWRITE_PARAMS
    try:
        for t in run.backward(gy.to(DEV))[:5]:
            t.fill_(0.25)
        got = run.backward(gy.to(DEV))[:5]
    finally:
        n.OVERWRITE_PARAMS = old
    for a, e in zip(got, want):
        assert_close(a, e.double().cpu() + (0.25 if accumulate else 0), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("shape,bs,batch,outer", [s for s in SHAPES if s[0][2] < 64],
                         ids=[i for i in ids if "x64-" not in i])
def test_gated_body(shape, bs, batch, outer):
    import torch.nn.functional as F

    from gridnet_amd import GatedGridnet, GridLayerNorm
    from gridnet_amd.network import gated_body
    from oracle.gated import gated_step_fast

    print(f"gated rows chain {shape} B={batch} outer={outer}", flush=True)
    gamma, beta, x, gy = inputs(shape, batch)
    (w0, b0, _), (w1, b1, _) = make_params(shape, seed=8), make_params(shape, seed=9)
    params = [torch.stack([w0, w1], 1), torch.stack([b0, b1]), gamma, beta]
    net = GatedGridnet(shape, 1, bs, device=DEV, activation="tanh")
    norm = GridLayerNorm(shape, device=DEV)
    with torch.no_grad():
        for p, t in zip((net.weight, net.bias, norm.weight, norm.bias), params):
            p.copy_(t)
    leaf = x.to(DEV).requires_grad_(True)
    y = gated_body(leaf, net, norm, outer)
    assert type(y.grad_fn).__name__ == "GatedBodyOpBackward"
    y.backward(gy.to(DEV), retain_graph=True)
    got = [y, leaf.grad, net.weight.grad, net.bias.grad, norm.weight.grad, norm.bias.grad]
    with torch.no_grad():
        assert torch.equal(gated_body(leaf, net, norm, outer), y)

    wide = [t.double().requires_grad_(True) for t in (x, *params)]
    h = wide[0]
    for _ in range(outer):
        h = F.layer_norm(gated_step_fast(wide[1], wide[2], h, 1, bs, "tanh"), shape, wide[3], wide[4])
    h.backward(gy.double())
    for name, a, e in zip(("y", "dx0", "dweight", "dbias", "dgamma", "dbeta"), got, [h, *[t.grad for t in wide]]):
        assert_close(a, e, rtol=2e-4, atol=2e-5, what=name)
    once = net.bias.grad.clone()
    y.backward(gy.to(DEV))  # the graph was kept
    assert torch.equal(net.bias.grad, 2 * once)
