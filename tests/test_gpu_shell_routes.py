"""Calls that the shell blocks are slow at go to the lane-per-peak kernel: many peaks per cell, and
peaks gathered to a large hunt radius, inside the tile and with balls that leave it.  The results
are the plain order's bit for bit, and the call takes no longer than half as much again as that
kernel with every peak's extent given (no crossing pass): it took 4.2, 2.1 and 1.9 times as long."""
import time

import pytest
import torch

from huntian_hip import api
from test_gpu_shell_blocks import _fields, _peaks, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nhunt,count,lo,fcrit", [
    (64, 8, 300_000, 9, None), (96, 45, 60_000, 0, -1e9), (256, 30, 100_000, 31, -1e9)])
def test_no_slower_than_a_lane_per_peak(websky, n, nhunt, count, lo, fcrit):
    f, pk = _fields(n, n, False), _peaks(n, count, n + 1, lo, n - lo)
    stab = api.build_shell_tables(nhunt)

    def run(order, **kw):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        r = api.shell_analyse(f, pk["pi"], pk["pj"], pk["pk"], pk["Rf"], pk["ir2min"], stab, websky,
                              alatt=2.0, ZZon=1.0, nbuff=lo, variant="C", order=order,
                              fcrit=api.fsc_of_z(websky, 0.0) if fcrit is None else fcrit, **kw)
        torch.cuda.synchronize()
        return r, time.perf_counter() - t0

    plain, _ = run("plain")
    got, _ = run("crossing")
    _same(got, plain, f"n {n} nhunt {nhunt}")
    extent = got["nshells_used"].clone()
    _same(run("given", extent=extent)[0], plain, "extents given")
    crossing = min(run("crossing")[1] for _ in range(4))
    given = min(run("given", extent=extent)[1] for _ in range(4))
    print(f"n {n} nhunt {nhunt}: {1e3 * crossing:.2f} ms, a lane per peak {1e3 * given:.2f}", flush=True)
    assert crossing < 1.5 * given


@pytest.mark.parametrize("n,nhunt,count", [
    (40, 2, 3000), (40, 3, 3000), (200, 3, 200), (200, 3, 8000), (200, 6, 20_000), (201, 4, 90_000)])
def test_small_hunt_radii(websky, n, nhunt, count):
    """On either side of the line between staged bricks and cell records."""
    f, pk = _fields(n, n, False), _peaks(n, count, 8)
    kw = dict(alatt=2.0, ZZon=1.0, fcrit=api.fsc_of_z(websky, 0.0), variant="C")
    arg = (f, pk["pi"], pk["pj"], pk["pk"], pk["Rf"], pk["ir2min"], api.build_shell_tables(nhunt),
           websky)
    _same(api.shell_analyse(*arg, order="crossing", **kw), api.shell_analyse(*arg, order="plain", **kw),
          f"n {n} nhunt {nhunt}")
