"""The shell analysis by shell blocks (crossing schedule of a direct call) against the
lane-per-peak kernel (plain order), every result field and the mask bit for bit, where the block
gather can go wrong: tiles whose rows are 16-byte aligned and not, peaks on the faces (balls that
leave the tile), hunt radii inside, at and beyond the bricks' 8-cell halo, a brick with more
peaks and more items than it takes at a time, few and many peaks (row and lane crossing passes),
sparse peaks (no bricks), uneven tiles with an empty one, non-finite field values."""
import numpy as np
import pytest
import torch

from huntian_hip import api, synth

pytestmark = pytest.mark.gpu


def _fields(n, seed, lapd):
    f, _ = synth.fields_torch(n, 2.0 * n, seed, "cuda")
    f = {k: api.to_device_field(v) for k, v in f.items()}
    if lapd:
        f["lapd"] = api.to_device_field(-2.0 * f["delta"])
    return f


def _peaks(n, count, seed, lo=0, hi=None):
    """Cells of the densest `count` of a random sample (no need to be maxima), with filters."""
    rng = np.random.default_rng(seed)
    hi = n if hi is None else hi
    c = rng.integers(lo, hi, (count, 3)) + 1
    Rf = rng.choice([1.5, 3.0, 6.0, 12.0, 20.0], count, p=[0.4, 0.3, 0.15, 0.1, 0.05])
    ir2 = np.array([api.ir2min_of(r, 2.0) for r in Rf], np.int32)
    t = [torch.as_tensor(np.ascontiguousarray(c[:, q]), dtype=torch.int32, device="cuda")
         for q in range(3)]
    return dict(pi=t[0], pj=t[1], pk=t[2], Rf=torch.as_tensor(Rf, device="cuda"),
                ir2min=torch.as_tensor(ir2, device="cuda"))


def _same(a, b, label):
    for k in a:
        x, y = a[k], b[k]
        eq = x == y
        if x.dtype == torch.float64:
            eq |= torch.isnan(x) & torch.isnan(y)
        assert bool(eq.all()), (label, k, int((~eq).sum()))


def _compare(fields, pk, n, nhunt, ct, variant, label, nbuff=0):
    stab = api.build_shell_tables(nhunt)
    out = []
    for order in ("crossing", "plain"):
        mask = api.fortran_empty((n, n, n), torch.int8)
        mask.zero_()
        r = api.shell_analyse(fields, pk["pi"], pk["pj"], pk["pk"], pk["Rf"], pk["ir2min"], stab, ct,
                              alatt=2.0, ZZon=1.0, fcrit=api.fsc_of_z(ct, 0.0), nbuff=nbuff,
                              variant=variant, mask=mask, order=order)
        out.append((r, mask))
    _same(out[0][0], out[1][0], label)
    assert torch.equal(out[0][1], out[1][1]), label
    halos = int((out[0][0]["RTHL"] > 0).sum())
    print(f"{label}: {len(pk['pi'])} peaks, {halos} halos", flush=True)
    return halos


@pytest.mark.parametrize("n,nhunt,count,variant,lapd", [
    (40, 3, 600, "C", False),     # no crossing for most; one block
    (48, 8, 2000, "A", True),     # the halo exactly; 16-byte rows
    (49, 9, 2000, "B", True),     # one cell beyond it; 4-byte rows
    (64, 12, 5000, "C", True),
    (80, 20, 9000, "C", False),
    (90, 40, 9000, "A", False),   # deep balls, many leaving the tile
    (64, 12, 40, "C", False),     # a few peaks: gathered from the fields
    (96, 10, 140_000, "C", False),  # the lane-per-peak crossing pass, 600 peaks per brick
])
def test_blocks_equal_lane_per_peak(websky, n, nhunt, count, variant, lapd):
    f = _fields(n, 7 * n, lapd)
    assert _compare(f, _peaks(n, count, n), n, nhunt, websky, variant, f"n {n} nhunt {nhunt}") > 0


def test_crowded_brick(websky):
    """Every cell of one brick a peak: more than 256 peaks and more items than fit at once."""
    n = 64
    f = _fields(n, 5, False)
    g = np.arange(16, 32) + 1
    c = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    pk = _peaks(n, len(c), 3)
    for q, key in enumerate(("pi", "pj", "pk")):
        pk[key] = torch.as_tensor(np.ascontiguousarray(c[:, q]), dtype=torch.int32, device="cuda")
    assert _compare(f, pk, n, 15, websky, "C", "crowded brick") > 0


def test_non_finite_and_subnormal_values(websky):
    n = 64
    f = _fields(n, 6, False)
    f["etax"][20:24, 30, 30] = float("inf")
    f["etay"][30, 20:24, 31] = float("nan")
    f["etaz"] = api.to_device_field(f["etaz"] * 1e-42)
    f["delta"][40, 40, 40] = float("nan")
    _compare(f, _peaks(n, 3000, 9), n, 10, websky, "C", "non-finite values")


def test_uneven_tiles_with_an_empty_one(websky):
    tiles = []
    for n, count in ((40, 900), (33, 0), (66, 5000), (48, 1)):
        t = dict(fields=_fields(n, n, False), **_peaks(n, count, n))
        tiles.append(t)
    stab = api.build_shell_tables(11)
    kw = dict(alatt=2.0, ZZon=1.0, fcrit=api.fsc_of_z(websky, 0.0))
    a = api.shell_analyse_tiles(tiles, stab, websky, order="crossing", **kw)
    b = api.shell_analyse_tiles(tiles, stab, websky, order="plain", **kw)
    for q, (x, y) in enumerate(zip(a, b)):
        _same(x, y, f"tile {q}")
