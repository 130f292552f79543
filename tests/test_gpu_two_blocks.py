"""The forward with two blocks to a workgroup (csrc/step_fast.hip, FwdThread) against the same samples in a batch whose
size takes the kernel with one: the same bits.  Which one a call takes: two_blocks() there, on 256 CUs."""

import pytest
import torch

from helpers import assert_close, make_acts, make_params
from test_gpu_fused_chain import run_chain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# just too many elements for the kernels of small grids, one to a workgroup, and one more than the chunks; blocks at
# both ends of a row; three chunks, the last one short (a walk of 24 iterations) against 88; more blocks than the chip
# holds (16 against 136)
@pytest.mark.parametrize("shape,two,one,inner,activation", [
    *[((16, 16, 64), 17, 600, 2, a) for a in ("relu", "leaky_relu", "silu", "tanh")], ((16, 16, 64), 49, 600, 3, "silu"),
    ((8, 24, 128), 11, 300, 3, "tanh"), ((64, 64, 64), 17, 64, 4, "silu"), ((128, 128, 128), 2, 17, 8, "leaky_relu")], ids=str)
def test_step_is_the_one_of_single_blocks(shape, two, one, inner, activation):
    from gridnet_amd import gridnet_step

    print(f"two blocks, step {shape} B={two}/{one} inner={inner} {activation}", flush=True)
    w, b, s = (t.to(DEV) for t in make_params(shape, seed=4))
    x = make_acts(max(two, one), shape, seed=6).to(DEV)
    both = min(two, one)
    y2, y1 = (gridnet_step(w, b, s, x[:n], inner, 8, 1e-5, False, activation) for n in (two, one))
    assert torch.isfinite(y2).all() and torch.equal(y2[:both], y1[:both])


# ... with the LayerNorm folded in, in pairs of elements (an odd batch) and one by one, and its statistics
@pytest.mark.parametrize("shape,two,one,inner,outer", [
    ((32, 32, 64), 9, 2, 2, 3), ((32, 64, 64), 4, 1, 5, 2), ((32, 32, 64), 75, 200, 2, 2), ((64, 64, 64), 17, 64, 4, 2),
    ((128, 128, 128), 1, 17, 8, 2)], ids=str)
def test_chain_is_the_one_of_single_blocks(shape, two, one, inner, outer):
    print(f"two blocks, chain {shape} B={two}/{one} inner={inner}", flush=True)
    both = min(two, one)
    (y2, s2), (y1, s1) = (run_chain(shape, n, inner, outer, False) for n in (two, one))
    for j in range(outer):
        assert torch.isfinite(y2[j]).all() and torch.equal(y2[j][:both], y1[j][:both]), f"y {j}"
        assert torch.equal(s2[j][:both], s1[j][:both]), f"stats {j}"


# ... and finishing the statistics of the step before: the same sums in double, in another order
@pytest.mark.parametrize("shape,batch,inner", [((32, 32, 64), 9, 2), ((32, 32, 64), 75, 2)], ids=str)
def test_chain_that_merges(shape, batch, inner):
    from gridnet_amd import native as n

    print(f"two blocks, merging {shape} B={batch}", flush=True)
    assert n.lib.gridnet_hip_fused_forward_chain_merges(n.F32, batch, *shape, inner, 8)
    got, want = (run_chain(shape, batch, inner, 3, merges) for merges in (True, False))
    for j in range(3):
        assert_close(got[1][j], want[1][j], rtol=2e-7 * (1 + 50 * j), atol=1e-7 * (1 + 50 * j), what=f"stats {j}")
        assert_close(got[0][j], want[0][j], rtol=1e-5, atol=1e-5, what=f"y {j}")
