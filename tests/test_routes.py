"""Which kernels a fused step takes: both sides of the rules that choose by size (256 compute units, as without a device)."""

import pytest

BLOCKS, ROWS, PAIRS, QUADS = range(4)


def route(shape, batch, inner, block_size, residual=0, backward=0, workspace=None):
    from gridnet_amd.native import lib

    if workspace is None:
        workspace = lib.gridnet_hip_fused_workspace_bytes(batch, *shape, inner, block_size, backward)
    return lib.gridnet_hip_fused_route(batch, *shape, inner, block_size, residual, backward, workspace)


# measured on either side, the slower kernel 3 to 70 % behind: few samples of few blocks for a chip, at most six to a CU; places of
# a wave that are mostly empty where the chip has more than five rounds of them; half empty, eight rounds and more workgroups than
# it holds
@pytest.mark.parametrize("shape,batch,inner,want", [
    ((16, 16, 36), 4, 2, BLOCKS), ((32, 32, 12), 6, 6, BLOCKS), ((64, 64, 4), 6, 4, BLOCKS), ((32, 32, 20), 4, 6, BLOCKS),
    ((32, 32, 20), 5, 2, QUADS), ((32, 32, 36), 5, 2, QUADS), ((64, 64, 20), 5, 4, QUADS), ((64, 64, 64), 128, 8, QUADS),
    ((64, 64, 4), 128, 8, BLOCKS), ((128, 128, 4), 33, 2, BLOCKS), ((128, 128, 4), 13, 8, BLOCKS),
    ((128, 128, 4), 12, 4, QUADS), ((64, 64, 4), 32, 8, QUADS), ((64, 64, 8), 128, 4, QUADS), ((128, 128, 20), 9, 4, QUADS),
    ((128, 128, 8), 33, 4, BLOCKS), ((128, 128, 8), 16, 4, QUADS), ((128, 128, 12), 64, 4, QUADS)], ids=str)
@pytest.mark.parametrize("residual", [0, 1])
def test_forward_of_small_blocks(shape, batch, inner, want, residual):
    assert route(shape, batch, inner, 4, residual) == want


# the backward: a walk of 32 at least, groups of four samples that are nearly full, half of the places of its waves taken, seven tenths
# where there are three rounds of them
@pytest.mark.parametrize("shape,batch,inner,want", [
    ((64, 64, 64), 8, 2, BLOCKS), ((64, 64, 64), 16, 2, QUADS), ((64, 64, 64), 5, 4, BLOCKS), ((64, 64, 64), 4, 8, QUADS),
    ((40, 40, 40), 32, 4, BLOCKS), ((44, 44, 44), 32, 4, QUADS), ((52, 52, 52), 32, 4, QUADS), ((64, 64, 64), 32, 9, BLOCKS),
    ((128, 56, 36), 100, 5, BLOCKS), ((56, 80, 52), 16, 6, BLOCKS), ((80, 80, 40), 20, 4, BLOCKS), ((80, 80, 48), 20, 4, QUADS)], ids=str)
def test_backward_of_small_blocks(shape, batch, inner, want):
    assert [route(shape, batch, inner, 4, residual, backward=1) for residual in (0, 1, 2)] == [want, want, BLOCKS]
