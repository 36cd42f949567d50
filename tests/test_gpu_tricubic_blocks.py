"""The tri-cubic interpolation by runs of cells, which tiles of 96 cells a side and more and of four
coarse cells and more take: every block side it has (4 to 32), whole against the oracle and the per-cell
kernel (tuning tricubic_tab = 0), bit for bit.  Sides at and beside multiples of the block, runs
that start at any cell, tiles that wrap around the grid many times, coarse grids down to one cell, an
output that is not 16-byte aligned."""
import numpy as np
import pytest
import torch

from huntian_hip import api
from oracle import fields as F

pytestmark = pytest.mark.gpu


def _shifted(n, dev, k=1):
    """Column-major n^3 outputs that start 4 bytes past an aligned address."""
    return [torch.empty(n ** 3 + 1, device=dev)[1:].view(n, n, n).permute(2, 1, 0) for _ in range(k)]


@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("block,M,tile,nsub,nmesh", [
    (4, 40, (1, 2, 1), 90, 96), (4, 1, (1, 1, 1), 96, 96), (4, 9, (3, 1, 2), 91, 97),
    (4, 33, (2, 2, 5), 95, 99), (8, 20, (2, 1, 3), 96, 96), (8, 2, (1, 4, 1), 83, 101),
    (8, 13, (3, 2, 1), 97, 104), (16, 8, (2, 1, 2), 90, 96), (16, 1, (1, 1, 2), 95, 98),
    (16, 7, (2, 3, 1), 85, 97), (32, 5, (2, 1, 1), 111, 128), (32, 3, (1, 2, 3), 117, 130)])
def test_runs_equal_the_oracle(monkeypatch, block, M, tile, nsub, nmesh, shifted):
    coarse = np.random.default_rng(block * 1000 + nmesh).standard_normal((M, M, M)).astype(np.float32)
    if shifted:
        monkeypatch.setattr(api, "_field_out", _shifted)
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
    assert (out[1].data_ptr() % 16 != 0) == shifted
    assert torch.equal(out[1], out[0])
    np.testing.assert_array_equal(out[1].cpu().numpy(),
                                  F.interpolate_to_tile(coarse, *tile, nsub, nmesh, M * block, M))
