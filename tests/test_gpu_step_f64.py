"""The fp64 step (csrc/step_f64.hip) against the CPU oracle in fp64.  Bound: 1e-9 as for every fp64 run; the
sums have at most 27 x 32 x batch terms of unit size, 1e-12 of rounding."""

import pytest
import torch

from helpers import acts_clear_of_kink, assert_close, make_acts, make_params
from test_gpu_step import compare, oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# inner iterations: the fewest; with 8^3 blocks the most whose activations are kept (10), one more, the most
# whose pre-activations are (15), one more (the scattering kernel); 4^3 blocks: three shell entries per thread;
# grids of one block (the whole shell outside the grid) and of several; batches that one workgroup walks and
# that are split; just below and above 1024 blocks (above and batch 1: the scattering kernel)
@pytest.mark.parametrize("normalize", [False, True], ids=["plain", "normalize"])
@pytest.mark.parametrize("shape,bs,inner,batch,activation", [
    ((8, 8, 8), 8, 1, 2, "silu"), ((8, 16, 24), 8, 3, 5, "tanh"), ((16, 8, 8), 8, 3, 1, "tanh"),
    ((8, 8, 16), 8, 10, 2, "silu"), ((8, 8, 16), 8, 11, 2, "silu"), ((24, 8, 16), 8, 15, 2, "tanh"),
    ((16, 8, 8), 8, 16, 2, "tanh"), ((48, 48, 48), 8, 2, 2, "silu"), ((4, 4, 4), 4, 2, 3, "silu"),
    ((8, 12, 20), 4, 4, 7, "relu"), ((4, 8, 12), 4, 32, 2, "tanh"), ((40, 40, 40), 4, 2, 2, "silu"),
    ((40, 40, 44), 4, 2, 2, "silu")])
def test_step_f64(shape, bs, inner, batch, activation, normalize):
    compare((shape, bs, inner, normalize, activation), dtype=torch.float64, rtol=1e-9, atol=1e-9, batch=batch)


@pytest.mark.parametrize("normalize", [0, 1], ids=["plain", "normalize"])
@pytest.mark.parametrize("share", ["all", "required", "none"])
@pytest.mark.parametrize("shape,batch", [((8, 16, 8), 4), ((16, 8, 8), 300)])
def test_workspaces_and_accumulation(shape, batch, share, normalize):
    """With all of the workspace, the part without room for copies of the gradients (the batch is not split)
    and none (the scattering kernel): the same to rounding, and without the overwrite flags everything is
    added to what is there.  Two runs with a workspace give the same bits."""
    from gridnet_amd import native as n

    w, b, r = make_params(shape, seed=3, dtype=torch.float64)
    x = make_acts(batch, shape, seed=4, dtype=torch.float64)
    gy = make_acts(batch, shape, seed=5, dtype=torch.float64)
    d = [t.to(DEV) for t in (w, b, r, x, gy)]
    dt = n.dtype_id(d[0])
    nbytes = n.lib.gridnet_hip_backward_workspace_bytes(dt, batch, *shape, 2, 8, normalize)
    if share != "all":
        cells = shape[0] * shape[1] * shape[2]
        up = lambda v: (v + 255) // 256 * 256
        nbytes = 0 if share == "none" else up(8 * batch * cells) + normalize * up(16 * batch * cells // 512)
    want = oracle(w, b, r, x, gy, 2, 8, 1e-5, bool(normalize), "silu")[1]
    for flags, preset in ((0, 0.25), (n.OVERWRITE, float("nan")), (n.OVERWRITE_PARAMS, 0.25)):
        runs = []
        for _ in range(2):
            grads = [torch.full_like(t, preset) for t in (d[0], d[1], d[2], d[3])]
            ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=DEV)
            n.check(n.lib.gridnet_hip_backward(
                dt, *(t.data_ptr() for t in d), *(g.data_ptr() for g in grads), batch, *shape, 2, 8, 1e-5,
                normalize, n.activation_id("silu"), flags, ws.data_ptr() if nbytes else None, nbytes,
                n.current_stream(d[0])))
            runs.append(grads)
        torch.cuda.synchronize()
        for name, g, again, e in zip(("dweight", "dbias", "dscale", "dx"), *runs, want):
            added = 0.0 if flags == n.OVERWRITE or flags and name != "dx" else preset
            assert_close(g, e + added, 1e-9, 1e-9, name)
            assert share == "none" or torch.equal(g, again), name


def test_infinity_stays_where_its_taps_are():
    """One infinite cell, on the face between two blocks: the same entries are finite as in the oracle."""
    from test_gpu_step import run_op

    shape = (16, 8, 8)
    w, b, r = make_params(shape, seed=7, dtype=torch.float64)
    x = make_acts(1, shape, seed=8, dtype=torch.float64)
    x[0, 8, 3, 0] = float("inf")
    gy = make_acts(1, shape, seed=9, dtype=torch.float64)
    _, grads = run_op(w, b, r, x, gy, 1, 8, 1e-5, False, "relu")
    want = oracle(w, b, r, x, gy, 1, 8, 1e-5, False, "relu")[1]
    for name, g, e in zip(("dweight", "dbias", "dscale", "dx"), grads, want):
        assert torch.equal(torch.isfinite(g), torch.isfinite(e)), name
    assert not torch.isfinite(grads[0]).all()


@pytest.mark.parametrize("shape,bs,inner,batch", [((24, 24, 24), 8, 3, 2), ((24, 24, 24), 8, 12, 3),
                                                  ((12, 12, 12), 4, 3, 3), ((12, 12, 12), 4, 8, 2)])
def test_a_window_far_from_zero_is_normalised_as_exactly(shape, bs, inner, batch):
    """The middle block of three a side, whose window holds no zeros from outside the grid, does not depend on a
    constant that every input has on top.  Here that is 2^20, on inputs of 30 bits behind the point, which it leaves
    exact.  Worked on without it the gradients are those of inputs around zero, to the bound there; one rounding at its
    scale is 1e-10.  (The output holds the constant: half an ulp of it.)"""
    from test_gpu_step import run_op

    w, b, r = make_params(shape, seed=13, dtype=torch.float64)
    x = torch.round(make_acts(batch, shape, seed=14, dtype=torch.float64) * 2 ** 30) / 2 ** 30
    middle = (..., *[slice(bs, 2 * bs)] * 3)
    gy = torch.zeros_like(x)
    gy[middle] = make_acts(batch, (bs, bs, bs), seed=15, dtype=torch.float64)
    y, grads = run_op(w, b, r, x + 2.0 ** 20, gy, inner, bs, 1e-5, True, "tanh")
    want_y, want = oracle(w, b, r, x, gy, inner, bs, 1e-5, True, "tanh")
    assert_close(y[middle].cpu() - 2.0 ** 20, want_y[middle], 0, 2.0 ** -32, "y")
    for name, g, e in zip(("dweight", "dbias", "dscale", "dx"), grads, want):
        part = middle if name != "dx" else (...,)
        assert_close(g[part], e[part], 1e-12, 1e-12, name)
