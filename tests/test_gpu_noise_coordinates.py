"""The noise kernel's coordinates on grids of more than 2^21 cells a side, whose linear indices pass
2^63: 32 bits wide below 2^31 cells a side, 64 above.  Cells of the tile, its corners, edges and
those wrapped around the grid, against the oracle's Gaussian of index i + N (j + N k) modulo 2^64 (one
Float32 ulp, as in the noise tests)."""
import itertools

import numpy as np
import pytest

from huntian_hip import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tile,nsub,nmesh", [
    ((1 << 22) + 6, (1, 1, 1), 10, 21), ((1 << 31) - 2, (1, 1, 1), 16, 21),
    ((1 << 31) - 1, (1, 2, 1), 15, 20), ((1 << 31), (1, 1, 2), 16, 22),
    ((1 << 31) + 2, (1, 1, 1), 16, 21), ((1 << 31) + 1, (2, 1, 3), 16, 18),
    ((1 << 40) + 4, (1, 1, 1), 11, 17), ((1 << 31) - 2, ((1 << 27) + 1, 1 << 27, 3), 16, 19)])
def test_cells_of_large_grids(oracle, N, tile, nsub, nmesh):
    seed = 5
    got = np.asarray(api.generate_tile_noise(*tile, nsub, nmesh, N, seed))
    start = [(t - 1) * nsub - (nmesh - nsub) // 2 for t in tile]
    rng = np.random.default_rng(nmesh)
    ends = [0, 1, (nmesh - nsub) // 2 - 1, (nmesh - nsub) // 2, nmesh - 2, nmesh - 1]
    cells = list(itertools.product(ends, repeat=3)) + rng.integers(0, nmesh, (300, 3)).tolist()
    worst = 0
    for c in cells:
        i, j, k = ((s + q) % N for s, q in zip(start, c))
        want = np.float32(oracle.threefry_gauss(seed, (i + N * (j + N * k)) % (1 << 64)))
        d = abs(int(got[tuple(c)].view(np.int32)) - int(want.view(np.int32)))
        worst = max(worst, d)
        assert d <= 1, (c, got[tuple(c)], want)
    print(f"N {N}: {len(cells)} cells, worst {worst} ulp", flush=True)

