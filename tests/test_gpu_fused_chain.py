"""gridnet_hip_fused_forward_chain: the forward of a chain whose steps finish the statistics of the step before
(csrc/step_fast.hip, MERGE), against the same steps one call at a time, which a kernel of its own finishes."""

import pytest
import torch

from helpers import assert_close, make_acts, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def run_chain(shape, batch, inner, outer, merges, separate=False, bs=8):
    from gridnet_amd import native as n

    g = torch.Generator().manual_seed(5)
    sets = [[t.to(DEV) for t in make_params(shape, seed=4 + j)] for j in range(outer if separate else 1)]
    sets = sets if separate else sets * outer
    gamma, beta = ((a + 0.2 * torch.randn(shape, generator=g)).to(DEV) for a in (1, 0))
    x = make_acts(batch, shape, seed=6).to(DEV)
    y = [torch.full_like(x, float("nan")) for _ in range(outer)]
    stats = [torch.full((batch, 2), float("nan"), device=DEV) for _ in range(outer)]
    dims = (batch, *shape)
    act, stream = n.activation_id("silu"), n.current_stream(x)
    if merges:
        nbytes = n.lib.gridnet_hip_fused_forward_chain_workspace_bytes(*dims, inner, bs)
        ws = n.workspace(nbytes, x.device)
        n.check(n.lib.gridnet_hip_fused_forward_chain(
            n.F32, *(n.pointers([p[k] for p in sets]) for k in range(3)), gamma.data_ptr(), beta.data_ptr(),
            x.data_ptr(), n.pointers(y), n.pointers(stats), *dims, inner, outer, bs, 1e-5, act, ws.data_ptr(), nbytes, stream))
    else:
        nbytes = n.lib.gridnet_hip_fused_workspace_bytes(*dims, inner, bs, 0)
        ws = n.workspace(nbytes, x.device)
        for j in range(outer):
            n.check(n.lib.gridnet_hip_fused_forward(
                n.F32, *(t.data_ptr() for t in sets[j]), gamma.data_ptr(), beta.data_ptr(),
                (y[j - 1] if j else x).data_ptr(), stats[j - 1].data_ptr() if j else None, y[j].data_ptr(),
                stats[j].data_ptr(), *dims, inner, bs, 1e-5, act, ws.data_ptr(), nbytes, stream))
    torch.cuda.synchronize()
    return y, stats


# one block and one sample; pairs of elements (an odd batch) and single ones; chunks that end early; more samples
# than a workgroup merges, more pairs than are worth merging (64^3, batch 40), 4^3 blocks and one inner iteration
# by whole rows (all three: a kernel of its own finishes the statistics)
@pytest.mark.parametrize("shape,batch,inner,outer,bs,merging", [
    ((8, 8, 8), 1, 2, 3, 8, True), ((16, 8, 24), 7, 2, 2, 8, True), ((32, 32, 32), 19, 2, 3, 8, True),
    ((32, 32, 32), 150, 2, 2, 8, True), ((8, 8, 8), 5000, 2, 2, 8, True), ((16, 16, 16), 1, 3, 1, 8, True),
    ((40, 48, 56), 5, 3, 3, 8, True), ((8, 8, 8), 120000, 1, 2, 8, False), ((64, 64, 64), 40, 1, 2, 8, False),
    ((8, 8, 16), 3, 2, 2, 4, False), ((16, 16, 32), 9, 1, 3, 8, False)], ids=str)
@pytest.mark.parametrize("separate", [False, True], ids=["shared", "separate"])
def test_chain_is_the_steps_one_after_the_other(shape, batch, inner, outer, bs, merging, separate):
    from gridnet_amd import native as n

    print(f"fused chain {shape} B={batch} inner={inner} outer={outer} bs={bs} separate={separate}", flush=True)
    assert bool(n.lib.gridnet_hip_fused_forward_chain_merges(n.F32, batch, *shape, inner, bs)) == merging
    got = run_chain(shape, batch, inner, outer, True, separate, bs)
    want = run_chain(shape, batch, inner, outer, False, separate, bs)
    for j, (a, e) in enumerate(zip(got[1], want[1])):  # the same sums in double, in another order
        assert_close(a, e, rtol=2e-7 * (1 + 50 * j), atol=1e-7 * (1 + 50 * j), what=f"stats {j}")
    for j, (a, e) in enumerate(zip(got[0], want[0])):
        assert_close(a, e, rtol=1e-5, atol=1e-5, what=f"y {j}")


def test_wrong_arguments_are_refused():
    from gridnet_amd import native as n

    x = torch.zeros(2, 8, 8, 8, device=DEV)
    w, b = torch.zeros(27, 8, 8, 8, device=DEV), torch.zeros(8, 8, 8, device=DEV)
    s = torch.zeros(2, 2, device=DEV)
    nbytes = n.lib.gridnet_hip_fused_forward_chain_workspace_bytes(2, 8, 8, 8, 2, 8)
    ws = n.workspace(nbytes, x.device)

    def call(outer=2, dtype=n.F32, nbytes=nbytes, bs=8, stats=(s, s.clone())):
        n.check(n.lib.gridnet_hip_fused_forward_chain(
            dtype, *(n.pointers([t] * 2) for t in (w, b, b)), b.data_ptr(), b.data_ptr(), x.data_ptr(),
            n.pointers([x.clone(), x.clone()]), n.pointers(stats), 2, 8, 8, 8, 2, outer, bs, 1e-5, 0, ws.data_ptr(), nbytes,
            n.current_stream(x)))

    for bad in (dict(outer=0), dict(dtype=1), dict(nbytes=nbytes - 1), dict(bs=5)):
        with pytest.raises(RuntimeError):
            call(**bad)
