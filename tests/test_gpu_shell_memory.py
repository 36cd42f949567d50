"""The shell analysis where the profiles of the shell blocks are large: many deep peaks in one 64^3
brick (their profiles together are half as large again as the 32 GiB a call may hold at a time),
and a device with too little memory left for them.  The call answers as the lane-per-peak kernel
(plain order) does, bit for bit, in the memory that kernel takes."""
import pytest
import torch

from huntian_hip import api
from test_gpu_shell_blocks import _fields, _peaks, _same

pytestmark = pytest.mark.gpu


def _run(f, pk, n, nhunt, ct, order):
    r = api.shell_analyse(f, pk["pi"], pk["pj"], pk["pk"], pk["Rf"], pk["ir2min"],
                          api.build_shell_tables(nhunt), ct, alatt=2.0, ZZon=1.0, fcrit=-1e9,
                          nbuff=nhunt, variant="C", order=order)
    print(order, n, nhunt, len(pk["pi"]), flush=True)
    return r


def test_crowded_brick_of_deep_peaks(websky):
    n, nhunt = 192, 20
    f, pk = _fields(n, 3, False), _peaks(n, 900_000, 4, 64, 128)
    plain = _run(f, pk, n, nhunt, websky, "plain")
    ctx = api.context(0)
    ctx.release_scratch()
    out = api.alloc_results(len(pk["pi"]))
    del out  # the results come from torch's cache, not from the memory measured
    free = torch.cuda.mem_get_info()[0]
    got = _run(f, pk, n, nhunt, websky, "crossing")
    used = free - torch.cuda.mem_get_info()[0]
    ctx.release_scratch()
    _same(got, plain, "crowded brick")
    # 84 blocks of 672 bytes a peak are 50.8e9; the budget and a quarter 42.9e9
    assert used < 44e9, used


def test_too_little_memory_for_the_profiles(websky):
    n, nhunt = 256, 8
    f, pk = _fields(n, 5, False), _peaks(n, 2_000_000, 6, 9, n - 9)
    plain = _run(f, pk, n, nhunt, websky, "plain")
    ctx = api.context(0)
    ctx.release_scratch()
    out = api.alloc_results(len(pk["pi"]))
    del out
    # the profiles take 14 blocks of 672 bytes a peak, 18.8e9 in all; the lane-per-peak kernel 2.6e9
    hog = torch.empty(torch.cuda.mem_get_info()[0] - 6_000_000_000, dtype=torch.uint8, device="cuda")
    try:
        got = _run(f, pk, n, nhunt, websky, "crossing")
    finally:
        del hog
        torch.cuda.empty_cache()
        ctx.release_scratch()
    _same(got, plain, "little memory")


def test_several_chunks_over_uneven_tiles(websky):
    """Profiles of more than the 32 GiB that a call holds at a time: chunks of the schedule that begin
    and end in the middle of tiles, every peak of every tile compared."""
    tiles = []
    for n, count in ((97, 100_000), (320, 7_000_000), (64, 40_000)):
        tiles.append(dict(fields=_fields(n, n, False), **_peaks(n, count, n, 9, n - 9)))
    tab = api.build_shell_tables(8)
    kw = dict(alatt=2.0, ZZon=1.0, fcrit=api.fsc_of_z(websky, 0.0))
    plain = api.shell_analyse_tiles(tiles, tab, websky, order="plain", **kw)
    ctx = api.context(0)
    ctx.release_scratch()
    got = api.shell_analyse_tiles(tiles, tab, websky, order="crossing", **kw)
    blocks = sum(float((r["nshells_used"].double() / 4).floor().sum()) + len(r["nshells_used"])
                 for r in got)
    ctx.release_scratch()
    print(f"{blocks * 672 / 2 ** 30:.1f} GiB of profiles", flush=True)
    assert blocks * 672 > 2 ** 35
    for q, (a, b) in enumerate(zip(got, plain)):
        _same(a, b, f"tile {q}")
