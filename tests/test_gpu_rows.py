"""The row-wise kernels on rows of other than 16, 32, 64 or 128 cells (csrc/cross_rows.hip and its
neighbours: every row takes a power of two of lanes, the spare ones idle), and on batches that are
split into chunks, against the CPU oracle in fp64 at the bar."""

import pytest
import torch

from helpers import assert_close, make_acts, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (grid, block, batch, inner): one lane short of a power of two, one over it, the smallest and the
# largest row; batches below and above the least number of elements a workgroup walks
SHAPES = [((8, 8, 8), 8, 1, 1), ((8, 16, 24), 8, 5, 1), ((4, 8, 12), 4, 2, 1), ((8, 8, 40), 4, 7, 1),
          ((8, 8, 56), 8, 3, 1), ((4, 4, 60), 4, 2, 1), ((8, 8, 72), 8, 2, 1), ((8, 8, 120), 8, 2, 2),
          ((16, 8, 24), 8, 4, 2), ((8, 16, 40), 8, 9, 2), ((8, 8, 36), 4, 3, 2), ((8, 8, 136), 8, 2, 2)]
ids = ["x".join(map(str, s)) + f"-{bs}-{b}-{i}" for s, bs, b, i in SHAPES]


@pytest.mark.parametrize("normalize", [False, True], ids=["plain", "normalize"])
@pytest.mark.parametrize("shape,bs,batch,inner", SHAPES, ids=ids)
def test_step(shape, bs, batch, inner, normalize):
    from gridnet_amd import gridnet_step
    from oracle.manual import gridnet_step_backward_manual
    from oracle.fast import gridnet_step_fast

    params, x, gy = make_params(shape, seed=1), make_acts(batch, shape, seed=2), make_acts(batch, shape, seed=3)
    leaves = [t.to(DEV).requires_grad_(True) for t in (*params, x)]
    y = gridnet_step(*leaves, inner, bs, 1e-5, normalize, "silu")
    y.backward(gy.to(DEV))
    wide = [t.double() for t in (*params, x)]
    assert_close(y, gridnet_step_fast(*wide, inner, bs, 1e-5, normalize, "silu"), what="y")
    want = gridnet_step_backward_manual(*wide, gy.double(), inner, bs, 1e-5, normalize, "silu")
    for name, leaf, exp in zip(("dweight", "dbias", "dscale", "dx"), leaves, want):
        assert_close(leaf.grad, exp, what=name)


@pytest.mark.parametrize("residual", [False, True], ids=["plain", "residual"])
@pytest.mark.parametrize("shape,bs,batch,inner", SHAPES, ids=ids)
def test_fused_chain(shape, bs, batch, inner, residual):
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    w, b, r = make_params(shape, seed=4)
    g = torch.Generator().manual_seed(5)
    gamma, beta = 1 + 0.2 * torch.randn(shape, generator=g), 0.2 * torch.randn(shape, generator=g)
    x, gy = make_acts(batch, shape, seed=6), make_acts(batch, shape, seed=7)
    outer = 2
    run = BodyRunner(*(t.to(DEV) for t in (w, b, r, gamma, beta)), batch, inner, outer, bs, "tanh",
                     fused=True, outer_residual=residual)
    got = [run.forward(x.to(DEV)).clone(), *run.backward(gy.to(DEV))]
    want = network_forward_backward([t.double() for t in (w, b, r, gamma, beta)], x.double(), gy.double(),
                                    inner_iterations=inner, outer_iterations=outer, block_size=bs,
                                    activation="tanh", outer_residual=residual)
    for name, a, e in zip(("y", "dweight", "dbias", "dscale", "dgamma", "dbeta", "dx0"), got, want):
        assert_close(a, e, rtol=2e-4, atol=2e-5, what=name)


@pytest.mark.parametrize("shape,bs,batch,inner", SHAPES, ids=ids)
def test_gated_step(shape, bs, batch, inner):
    from gridnet_amd import gated_gridnet_step
    from oracle.gated import gated_step_fast

    (w0, b0, _), (w1, b1, _) = make_params(shape, seed=8), make_params(shape, seed=9)
    w, b = torch.stack([w0, w1], 1), torch.stack([b0, b1])
    x, gy = make_acts(batch, shape, seed=10), make_acts(batch, shape, seed=11)
    results = []
    for leaves, f, g in (([t.to(DEV) for t in (w, b, x)], gated_gridnet_step, gy.to(DEV)),
                         ([t.double() for t in (w, b, x)], gated_step_fast, gy.double())):
        leaves = [t.requires_grad_(True) for t in leaves]
        y = f(*leaves, inner, bs, "tanh")
        y.backward(g)
        results.append([y, *[t.grad for t in leaves]])
    for name, a, e in zip(("y", "dweight", "dbias", "dx"), *results):
        assert_close(a, e, what=name)


# Grids of about one round of workgroups: the rule that gives rows of more than 64 cells to the kernel
# by rows or to the one by blocks, and chunks made shorter to even the rounds.  Samples do not mix, so
# a batch has to give what its samples give in twos; the first two are held against the oracle.
@pytest.mark.parametrize("residual", [False, True], ids=["plain", "residual"])
@pytest.mark.parametrize("shape,bs,batch,inner", [((48, 64, 96), 8, 4, 1), ((40, 48, 72), 8, 9, 1),
                                                  ((48, 88, 88), 8, 37, 1), ((80, 80, 72), 8, 33, 2),
                                                  ((52, 52, 52), 4, 21, 2)])
def test_rounds(shape, bs, batch, inner, residual):
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    w, b, r = make_params(shape, seed=12)
    g = torch.Generator().manual_seed(13)
    params = [w, b, r, 1 + 0.2 * torch.randn(shape, generator=g), 0.2 * torch.randn(shape, generator=g)]
    x = make_acts(batch, shape, seed=14)

    def forward(rows):
        run = BodyRunner(*(t.to(DEV) for t in params), len(rows), inner, 2, bs, "silu", fused=True,
                         backward=False, outer_residual=residual)
        return run.forward(rows.to(DEV)).cpu()

    got = forward(x)
    for i in range(0, batch, 2):
        assert_close(got[i:i + 2], forward(x[i:i + 2]), what=f"samples from {i}")
    want = network_forward_backward([t.double() for t in params], x[:2].double(), x[:2].double(),
                                    inner_iterations=inner, outer_iterations=2, block_size=bs,
                                    activation="silu", outer_residual=residual)[0]
    assert_close(got[:2], want, rtol=2e-4, atol=2e-5, what="y")
