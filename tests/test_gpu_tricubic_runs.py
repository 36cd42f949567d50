"""The tri-cubic interpolation by runs of cells (power-of-two blocks of 4 to 32 cells, tiles of four
coarse cells a side and more) against the per-cell kernel (tuning tricubic_tab = 0) bit for bit, and
against the oracle where it is quick: sides at and beside multiples of the block, runs that start
anywhere in the tile (stores of single cells), tiles that wrap around the grid, tiny coarse grids."""
import numpy as np
import pytest

from huntian_hip import api
from oracle import fields as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block,M,tile,nsub,nmesh", [
    (4, 16, (1, 1, 1), 16, 16), (4, 16, (4, 2, 1), 14, 17), (4, 9, (1, 3, 2), 12, 33),
    (4, 1, (1, 1, 1), 16, 16), (8, 2, (1, 2, 1), 16, 32), (8, 8, (3, 1, 2), 20, 37),
    (16, 8, (2, 1, 2), 48, 64), (16, 6, (1, 2, 1), 57, 70), (32, 6, (1, 1, 2), 96, 128),
    (32, 5, (2, 1, 1), 111, 131), (2, 16, (1, 1, 1), 16, 32), (16, 8, (1, 1, 1), 48, 63)])
def test_runs_equal_cells(block, M, tile, nsub, nmesh):
    import torch

    rng = np.random.default_rng(block * 1000 + nmesh)
    coarse = rng.standard_normal((M, M, M)).astype(np.float32)
    ctx = api.context(0)
    out = {}
    try:
        for tab in (1, 0):
            ctx.set_tuning(tricubic_tab=tab)
            out[tab] = api.interpolate_to_tile_gpu(coarse, *tile, nsub, nmesh, M * block, M,
                                                   return_device=True)
            print("tab", tab, block, M, nmesh, flush=True)
    finally:
        ctx.set_tuning(tricubic_tab=1)
    assert torch.equal(out[1], out[0])
    if nmesh <= 40:
        np.testing.assert_array_equal(out[1].cpu().numpy(),
                                      F.interpolate_to_tile(coarse, *tile, nsub, nmesh, M * block, M))
