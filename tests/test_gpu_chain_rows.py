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


@pytest.mark.parametrize("gated", [False, True], ids=["plain", "gated"])
def test_old_contents_are_added_once_to_the_finished_sum(gated):
    """A running sum that starts from the old contents rounds once per element; added to the finished
    sum they cost one rounding, so the result is exactly fp32(old + sum).  (Batch 5 is not split.)"""
    from gridnet_amd import native as n

    shape, batch = (8, 8, 32), 5
    gamma, beta, x, gy = (t.to(DEV) for t in inputs(shape, batch))
    w, b, r = (t.to(DEV) for t in make_params(shape, seed=4))
    if gated:
        w, b = torch.stack([w, w.flip(0)], 1), torch.stack([b, r])
    saved = torch.empty(3 if gated else 1, *x.shape, device=DEV)
    y_raw, out, dx, stats = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x), torch.empty(batch, 2, device=DEV)
    scale = None if gated else r.data_ptr()
    sizes = (batch, *shape, int(gated), 1)
    ws = n.workspace(max(n.lib.gridnet_hip_rows_chain_workspace_bytes(*sizes, d) for d in (0, 1)), DEV)
    n.check(n.lib.gridnet_hip_rows_chain_forward(
        w.data_ptr(), b.data_ptr(), scale, gamma.data_ptr(), beta.data_ptr(), x.data_ptr(), y_raw.data_ptr(),
        stats.data_ptr(), saved.data_ptr(), out.data_ptr(), batch, *shape, 1, int(gated), 1e-5,
        n.activation_id("tanh"), ws.data_ptr(), ws.numel(), n.current_stream(x)))

    def gradients(flags, into):
        dw, db, dr, dg, dbt = (t.data_ptr() for t in into)
        n.check(n.lib.gridnet_hip_rows_chain_backward(
            w.data_ptr(), scale, gamma.data_ptr(), beta.data_ptr(), x.data_ptr(), y_raw.data_ptr(), stats.data_ptr(),
            saved.data_ptr(), gy.data_ptr(), dw, db, None if gated else dr, dg, dbt, dx.data_ptr(), batch, *shape, 1,
            int(gated), n.activation_id("tanh"), flags, ws.data_ptr(), ws.numel(), n.current_stream(x)))
        return into

    like = (w, b, r, gamma, beta)
    alone = gradients(n.OVERWRITE_PARAMS, [torch.zeros_like(t) for t in like])
    old = [torch.randn(t.shape, generator=torch.Generator().manual_seed(9)).to(DEV) for t in like]
    got = gradients(0, [t.clone() for t in old])
    for name, a, o, g in zip(("dweight", "dbias", "dscale", "dgamma", "dbeta"), got, old, alone):
        assert torch.equal(a, o + g), name


def test_a_chain_adds_each_steps_sum_once():
    """dbeta of two steps where the second one's gradient is over 1e3 times the first one's: the first step's
    terms, sequentially summed, are added to the second's in ONE rounding, half an ulp of the result;
    term by term they would cost one each, fifteen of them.  (256 tubes: the batch is not split.)"""
    from gridnet_amd.runner import BodyRunner
    from oracle.network import network_forward_backward

    shape, batch = (64, 64, 16), 15
    gamma, beta, x, gy = inputs(shape, batch)
    w, b, r = make_params(shape, seed=4)
    params = [1e-6 * w, b, 1e5 * r, gamma, beta]  # the raw output varies by the biases, 1e4 times the input
    run = BodyRunner(*(t.to(DEV) for t in params), batch, 1, 2, 8, "silu", fused=True, forward_all=False)
    assert run.rows
    run.forward(x.to(DEV))
    got = run.backward(gy.to(DEV))[4].cpu()
    want = network_forward_backward([t.double() for t in params], x.double(), gy.double(), inner_iterations=1,
                                    outer_iterations=2, block_size=8, activation="silu")[5]
    last = torch.zeros(shape)
    for g in gy:  # the kernel's own order
        last = last + g
    first = want - gy.double().sum(0)
    assert first.abs().max() < 1e-2
    total = last.double() + first
    # one rounding, and what fp32 leaves on the first step's gradient
    bound = 2.0 ** -24 * total.abs() + 2e-4 * first.abs() + 1e-9
    off = (got.double() - total).abs()
    assert (off <= bound).all(), f"{int((off > bound).sum())} of {off.numel()}, worst {(off / bound).max():.1f} bounds"


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_gated_chain_at_the_scripts_defaults_is_as_exact_as_torch(seed):
    """32^3, batch 256, 64 steps, the gradient from the last layer only: against the same chain in fp64
    by torch's operators, this one and torch's own in fp32.  How well such a chain is conditioned
    depends on its parameters (over seeds both are between 2e-7 and 1e-2 off in the gradients), so what
    is held is the ratio: two evaluations in fp32, each a random share of the same bound, are seldom four
    times apart in norm.  1e-7: the rounding of the result itself, 6e-8 at most, on either side."""
    import torch.nn.functional as F

    from gridnet_amd import GatedGridnet, GridLayerNorm
    from gridnet_amd.network import gated_body
    from oracle.gated import gated_step_fast

    shape, batch, outer = (32, 32, 32), 256, 64
    print(f"gated chain against fp64, seed {seed}", flush=True)
    rnd = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*size, mean=0.0, std=1.0):
        return torch.randn(*size, generator=rnd, device=DEV) * std + mean

    params = [normal(27, 2, *shape, std=27 ** -0.5), normal(2, *shape, std=0.1), normal(*shape, mean=1.0, std=0.1),
              normal(*shape, std=0.1)]
    x = normal(*shape)[None].repeat(batch, 1, 1, 1)
    x[..., 0] = torch.rand(batch, *shape[:2], generator=rnd, device=DEV)
    gy = torch.zeros_like(x)
    gy[..., -1] = normal(batch, *shape[:2], std=1e-4)

    def by_torch(dtype):
        leaves = [t.to(dtype).requires_grad_(True) for t in (x, *params)]
        h = leaves[0]
        for _ in range(outer):
            h = F.layer_norm(gated_step_fast(leaves[1], leaves[2], h, 1, 8, "tanh"), shape, leaves[3], leaves[4])
        h.backward(gy.to(dtype))
        return [h.detach().double(), *[t.grad.double() for t in leaves]]

    net = GatedGridnet(shape, 1, 8, device=DEV, activation="tanh")
    norm = GridLayerNorm(shape, device=DEV)
    with torch.no_grad():
        for p, t in zip((net.weight, net.bias, norm.weight, norm.bias), params):
            p.copy_(t)
    leaf = x.clone().requires_grad_(True)
    y = gated_body(leaf, net, norm, outer)
    y.backward(gy)
    got = [y.detach(), leaf.grad, net.weight.grad, net.bias.grad, norm.weight.grad, norm.bias.grad]
    exact = by_torch(torch.float64)
    for name, a, t, e in zip(("y", "dx0", "dweight", "dbias", "dgamma", "dbeta"), got, by_torch(torch.float32), exact):
        ours, theirs = (((v.double() - e).norm() / e.norm()).item() for v in (a, t))
        print(f"  {name}: {ours:.2e} off, torch {theirs:.2e}", flush=True)
        assert ours <= 4 * theirs + 1e-7, name


# pairs of the merge: an odd number (a kernel of its own), two, more than a request's worth per thread, several
# threads to a sample and one; chunks that end early; too many samples per workgroup
# (backward: chunks of 32 samples, the most that the plain kernel merges for, of 33, 64 and 65)
@pytest.mark.parametrize("shape,batch", [((12, 12, 16), 5), ((4, 8, 16), 7), ((16, 16, 32), 37), ((32, 32, 32), 70),
                                         ((8, 8, 32), 300), ((16, 32, 64), 11), ((4, 4, 32), 5000),
                                         ((16, 16, 32), 1024), ((16, 16, 32), 1025), ((16, 16, 32), 2048),
                                         ((16, 16, 32), 2049)], ids=str)
def test_statistics_merged_by_the_next_step(shape, batch):
    """Statistics and backward sums of every step, against sums over the tensors themselves in double (fp32
    pairs over 256 values: 2^-24 times a few)."""
    from gridnet_amd.runner import BodyRunner

    print(f"merged statistics {shape} B={batch}", flush=True)
    gamma, beta, x, gy = inputs(shape, batch)
    run = BodyRunner(*(t.to(DEV) for t in (*make_params(shape, seed=4), gamma, beta)), batch, 1, 3, 4, "silu", fused=True,
                     forward_all=False, rows=True)
    y = run.forward(x.to(DEV)).clone()
    raw = run.s_all.double().flatten(2)
    mean, var = raw.mean(2), raw.var(2, unbiased=False)
    assert_close(run.stats[..., 0], mean, rtol=1e-6, atol=1e-6, what="mean")
    assert_close(run.stats[..., 1], (var + run.ln_eps).rsqrt(), rtol=1e-6, atol=0, what="rstd")
    last = (run.s_all[2] - run.stats[2, :, 0].view(-1, 1, 1, 1)) * run.stats[2, :, 1].view(-1, 1, 1, 1)
    assert_close(y, (last * run.gamma + run.beta).double(), rtol=1e-6, atol=1e-6, what="y")
    dx = run.backward(gy.to(DEV))[-1].clone()
    assert torch.equal(run.backward(gy.to(DEV))[-1], dx)
    # the first step's input gradient from the second's: backward once more in one step of its own
    step = BodyRunner(*(t.to(DEV) for t in (*make_params(shape, seed=4), gamma, beta)), batch, 1, 1, 4, "silu", fused=True,
                      forward_all=False, rows=True)
    h, grad = [x.to(DEV)], gy.to(DEV)
    for _ in range(2):
        h.append(step.forward(h[-1]).clone())
    for j in (2, 1, 0):  # every step's LayerNorm sums by the kernel for the last one
        step.forward(h[j])
        grad = step.backward(grad)[-1].clone()
    assert_close(dx, grad.double(), rtol=1e-5, atol=1e-5, what="dx")


@pytest.mark.parametrize("gated", [False, True], ids=["plain", "gated"])
def test_merged_sums_stay_in_the_workgroup(gated):
    """What a workgroup merges it hands to its waves through its LDS.  In memory, where all workgroups of a step would
    write the same words and read them back, the sums of the last step still stand after the backward."""
    from gridnet_amd import native as n

    shape, batch, outer = (16, 16, 32), 37, 3
    gamma, beta, x, gy = (t.to(DEV) for t in inputs(shape, batch))
    w, b, r = (t.to(DEV) for t in make_params(shape, seed=4))
    if gated:
        w, b = torch.stack([w, w.flip(0)], 1), torch.stack([b, r])
    sets, act, stream = 1 + gated, n.activation_id("tanh"), n.current_stream(x)
    saved = torch.empty(outer, 3 if gated else 1, *x.shape, device=DEV)
    y_raw, stats = torch.empty(outer, *x.shape, device=DEV), torch.empty(outer, batch, 2, device=DEV)
    out, dx = torch.empty_like(x), torch.empty_like(x)
    grads = [torch.empty_like(t) for t in (w, b, r, gamma, beta)]
    scale = None if gated else r.data_ptr()
    ws = n.workspace(max(n.lib.gridnet_hip_rows_chain_workspace_bytes(batch, *shape, int(gated), 1, d) for d in (0, 1)), DEV)
    n.check(n.lib.gridnet_hip_rows_chain_forward(
        w.data_ptr(), b.data_ptr(), scale, gamma.data_ptr(), beta.data_ptr(), x.data_ptr(), y_raw.data_ptr(),
        stats.data_ptr(), saved.data_ptr(), out.data_ptr(), batch, *shape, outer, int(gated), 1e-5, act,
        ws.data_ptr(), ws.numel(), stream))
    dw, db, dr, dg, dbt = (t.data_ptr() for t in grads)
    n.check(n.lib.gridnet_hip_rows_chain_backward(
        w.data_ptr(), scale, gamma.data_ptr(), beta.data_ptr(), x.data_ptr(), y_raw.data_ptr(), stats.data_ptr(),
        saved.data_ptr(), gy.data_ptr(), dw, db, None if gated else dr, dg, dbt, dx.data_ptr(), batch, *shape, outer,
        int(gated), act, n.OVERWRITE_PARAMS, ws.data_ptr(), ws.numel(), stream))
    want = torch.empty(batch, 2, device=DEV)
    scratch = n.workspace(n.lib.gridnet_hip_layernorm_workspace_bytes(0, batch, x[0].numel()), DEV)
    n.check(n.lib.gridnet_hip_layernorm_backward_sums(
        0, gy.data_ptr(), y_raw[-1].data_ptr(), stats[-1].data_ptr(), gamma.data_ptr(), want.data_ptr(), batch,
        x[0].numel(), scratch.data_ptr(), scratch.numel(), stream))
    # the workspace: two arrays of pairs, one for each wave and sample, and the sums behind them
    pairs = shape[0] // 4 * (shape[1] // 4) * (16 * shape[2] * sets // 2 // 64)
    at = -ws.data_ptr() % 256 + 2 * ((batch * pairs * 8 + 255) // 256 * 256)
    assert torch.equal(ws[at:at + batch * 8].view(torch.float32).view(batch, 2), want)
    assert torch.isfinite(dx).all()
