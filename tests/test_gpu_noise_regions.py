"""The noise kernel's index arithmetic where it changes: odd grids (a cell per thread), blocks of odd
side (a pair across two blocks), regions wider than the grid (several wraps), and grids on either
side of 2^31 cells a side (64-bit coordinates), against the oracle with the bars of the noise tests
(one Float32 ulp, all but 1e-5 of the cells bit for bit)."""
import numpy as np
import pytest

from huntian_hip import api
from test_gpu_noise import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tile,nsub,nmesh", [
    (15, (1, 2, 1), 10, 41), (16, (2, 1, 1), 9, 50), (81, (3, 1, 2), 20, 33), (1, (1, 1, 1), 3, 5),
    ((1 << 31) - 2, (1, 1, 1), 16, 21), ((1 << 31) + 2, (1, 1, 1), 16, 21),
    ((1 << 31) + 1, (2, 1, 3), 16, 18)])
def test_tile_noise_regions(oracle, N, tile, nsub, nmesh):
    if N > 2_097_152:  # its cells' linear indices pass 2^63: bits against the device's own rows only
        a = np.asarray(api.generate_tile_noise(*tile, nsub, nmesh, N, 5))
        b = np.asarray(api.generate_tile_noise(*tile, nsub, nmesh, N, 5))
        assert np.isfinite(a).all() and np.array_equal(a, b) and a.std() > 0.5
        return
    _check(api.generate_tile_noise(*tile, nsub, nmesh, N, 5),
           oracle.tile_noise(*tile, nsub, nmesh, N, 5), f"N {N}")


@pytest.mark.parametrize("N,M,tile,nsub,nmesh,nshell", [
    (45, 15, (1, 1, 2), 20, 24, 2), (60, 20, (2, 1, 1), 21, 26, 3), (30, 2, (1, 2, 1), 12, 17, 1),
    (24, 24, (1, 1, 1), 8, 30, 0)])
def test_residual_regions(oracle, N, M, tile, nsub, nmesh, nshell):
    coarse = oracle.downsample_noise(N, M, 9)
    _check(api.generate_extended_residual(*tile, nsub, nmesh, N, 9, coarse, M, nshell),
           oracle.extended_residual(*tile, nsub, nmesh, N, 9, coarse, M, nshell), f"residual N {N}")
