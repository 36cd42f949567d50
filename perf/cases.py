"""Workloads of the halo-finding path, as a program that uses it runs them.

Kinds of case (`case["op"]`):
  shell     radial-shell collapse of every candidate of one tile (api.shell_analyse): the mask
            is cleared and the analysis run, as the tile driver does after peak finding
  tiles     the same for several uneven tiles in one call (api.shell_analyse_tiles)
  peaks     multi-filter peak finding on smoothed fields (api.peak_find)
  bank      filter-bank smoothing and peak finding from the raw tile (api.peak_find_tile)
  convolve  isolated convolution of a tile's noise into delta and psi_1
            (api.isolated_convolve_gpu_multi)
  lpt       periodic 2LPT displacements and Laplacian of a tile (api.compute_2lpt_gpu,
            api.compute_laplacian_gpu)
  coarse    a tile's residual noise and the tri-cubic interpolation of the coarse delta and
            psi_1 onto it (api.generate_extended_residual, api.interpolate_to_tile_gpu)
  catalog   Lagrangian merge of a halo catalog with volume reduction, then its Eulerian
            positions and velocities (api.merge_catalog, api.finalize_eulerian)
Inputs are synthesised as the benchmark's are (Gaussian fields with the BBKS spectrum, cells
of 2 Mpc/h, thresholds of 1.5, collapse at z = 0).  A tile's candidates are capped at a number
a little below what its peak finding gives (the max_peaks of the tile driver), so that a case
has outputs of one size whatever the noise.
"""
import math
import os
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, "huntian.jl_amd"))

from huntian_hip import api, cosmology, synth  # noqa: E402
from huntian_hip.homeltab import WEBSKY_TABLE, read_homeltab  # noqa: E402

ALATT = 2.0
DEV = "cuda"
OBS = (0.0, 0.0, -2000.0)


def listed():
    return [
        # one small tile: a test run or an interactive look; launches and host work count
        dict(name="shell_n40", op="shell", n=40, nbuff=9, nhunt=8, nfilt=4, rmax=10.0,
             peaks=200, variant="C"),
        # the 128^3 tile the bracket network is trained on
        dict(name="shell_n128", op="shell", n=128, nbuff=16, nhunt=15, nfilt=16, rmax=20.0,
             peaks=24_000, variant="C"),
        # the 512^3 production tile
        dict(name="shell_n512", op="shell", n=512, nbuff=32, nhunt=20, nfilt=16, rmax=20.0,
             peaks=2_560_000, variant="C"),
        # the 1024^3 headline tile
        dict(name="shell_n1024", op="shell", n=1024, nbuff=64, nhunt=30, nfilt=24, rmax=34.0,
             peaks=21_000_000, variant="C"),
        # a batch of uneven tiles in one call (sides and buffers as the batched benchmark's)
        dict(name="tiles_24", op="tiles", sides="128 96 192 256 96 128 192 128 256 96 128 192 "
             "96 128 256 192 128 96 192 128 96 256 128 192", nbuff=20, nhunt=15, nfilt=16,
             rmax=20.0, variant="C"),
        # peak finding alone, on fields smoothed elsewhere
        dict(name="peaks_n512", op="peaks", n=512, nbuff=32, nfilt=16, rmax=20.0,
             peaks=2_560_000),
        # tile driver's peak finding of a small tile whose side is no power of two, with d2Rf
        dict(name="bank_n192", op="bank", n=192, nbuff=24, nfilt=16, rmax=20.0, wsmooth=1,
             lapd=True, peaks=75_000),
        # the same of the headline tile
        dict(name="bank_n1024", op="bank", n=1024, nbuff=64, nfilt=24, rmax=34.0, wsmooth=1,
             lapd=False, peaks=21_000_000),
        # long- and short-range fields of a 256^3 tile, padded to 512^3
        dict(name="convolve_n256", op="convolve", n=256, nshell=0),
        # second-order displacements and Laplacian of the 512^3 tile
        dict(name="lpt_n512", op="lpt", n=512),
        # noise and large-scale fields of a 256^3 tile of a 1024^3 grid
        dict(name="coarse_n256", op="coarse", nmesh=256, nsub=192, block=16, M=64, tile=3),
        # the catalog of a large tile
        dict(name="catalog_2M", op="catalog", halos=2_000_000, nf=33),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_side(rng, lo, hi):
    """An even side with no prime factor above 5 (what a user gives an FFT)."""
    ok = []
    for n in range(lo, hi + 1, 2):
        q = n
        for p in (2, 3, 5):
            while q % p == 0:
                q //= p
        if q == 1:
            ok.append(n)
    x = rng.uniform(math.log(lo), math.log(hi))
    return min(ok, key=lambda n: abs(math.log(n) - x))


def _cap(n, nbuff, nfilt):
    """Candidates of a tile: about one cell of the inner cube in 33.5 + 62 / nfilt, less 15 %
    and what the number scatters by in a small volume."""
    m = n - 2 * nbuff
    return max(1, int((0.85 - min(0.4, 13.0 / m)) * m ** 3 / (33.5 + 62.0 / nfilt)))


def draw(rng):
    op = rng.choice(["shell", "shell", "shell", "tiles", "peaks", "bank", "bank", "convolve",
                     "lpt", "coarse", "catalog"])
    nfilt = rng.randint(2, 16)
    rmax = round(rng.uniform(6.0, 24.0), 2)
    variant = rng.choice("CCAB")
    if op == "shell":
        n = _log(rng, 40, 320)
        nhunt = rng.randint(6, min(20, n // 5))
        nbuff = nhunt + rng.randint(1, 2)
        return dict(op=op, n=n, nbuff=nbuff, nhunt=nhunt, nfilt=nfilt, rmax=rmax,
                    peaks=_cap(n, nbuff, nfilt), variant=variant)
    if op == "tiles":
        sides = [str(_log(rng, 48, 200)) for _ in range(rng.randint(2, 12))]
        nhunt = rng.randint(6, 15)
        return dict(op=op, sides=" ".join(sides), nbuff=nhunt + 1, nhunt=nhunt, nfilt=nfilt,
                    rmax=rmax, variant=variant)
    if op == "peaks":
        n = _log(rng, 40, 400)
        nbuff = rng.randint(1, n // 6)
        return dict(op=op, n=n, nbuff=nbuff, nfilt=nfilt, rmax=rmax, peaks=_cap(n, nbuff, nfilt))
    if op == "bank":
        n = _smooth_side(rng, 40, 512)
        nbuff = rng.randint(1, n // 6)
        return dict(op=op, n=n, nbuff=nbuff, nfilt=nfilt, rmax=rmax,
                    wsmooth=rng.choice([0, 1, 1]), lapd=rng.random() < 0.4,
                    peaks=_cap(n, nbuff, nfilt))
    if op == "convolve":
        n_in = _smooth_side(rng, 24, 288)
        nshell = rng.choice([0, 0, 4, 6])
        return dict(op=op, n=n_in - 2 * nshell, nshell=nshell)
    if op == "lpt":
        return dict(op=op, n=_smooth_side(rng, 32, 480))
    if op == "coarse":
        nmesh = _log(rng, 40, 320)
        block = rng.choice([2, 3, 4, 5, 6, 8, 16, 16])
        M = max(8, 2 * nmesh // block)
        nsub = nmesh - 2 * rng.randint(0, nmesh // 8)
        return dict(op=op, nmesh=nmesh, nsub=nsub, block=block, M=M, tile=rng.randint(1, 3))
    return dict(op=op, halos=_log(rng, 1000, 2_000_000), nf=rng.choice([11, 33]))


# ---------------------------------------------------------------- inputs

def _radii(case):
    return synth.filter_radii(1.5, case["rmax"], case["nfilt"])


def _tile(n, nbuff, radii, peaks, seed):
    """A tile's fields and the first `peaks` candidates a driver's peak finding gives for it."""
    fields, dk = synth.fields_torch(n, n * ALATT, seed, DEV)
    mask = api.to_device_field(torch.zeros((n, n, n), dtype=torch.int8, device=DEV),
                               dtype=torch.int8)
    cols = []
    for q, R in enumerate(radii):
        f = api.to_device_field(synth.smooth_tophat_torch(dk, n, n * ALATT, R))
        pk = api.peak_find([f], [1.5], nbuff, mask, capacity=max(1024, (n - 2 * nbuff) ** 3 // 8))
        cols.append((pk["i"].clone(), pk["j"].clone(), pk["k"].clone(),
                     torch.full_like(pk["i"], R, dtype=torch.float64),
                     torch.full_like(pk["i"], api.ir2min_of(R, ALATT))))
        del f, pk
    del dk
    mask.zero_()
    keys = ("pi", "pj", "pk", "Rf", "ir2min")
    t = {key: torch.cat([c[q] for c in cols]) for q, key in enumerate(keys)}
    pick = torch.arange(peaks, device=DEV) % len(t["pi"])
    t = {key: v[pick] for key, v in t.items()}
    t.update(fields={k: api.to_device_field(v) for k, v in fields.items()}, mask=mask)
    return t


def _records(halos, nf, seed):
    """A raw catalog: clustered Lagrangian positions (Mpc/h) at the number density of the
    headline tile, radii log-normal about 3 Mpc/h, 1LPT and 2LPT displacements."""
    g = torch.Generator().manual_seed(seed)
    box = (halos / 2.3e-3) ** (1.0 / 3.0)
    nclus = max(1, halos // 20)
    centre = torch.rand((nclus, 3), generator=g) * box
    which = torch.randint(0, nclus, (halos,), generator=g)
    pos = centre[which] + 8.0 * torch.randn((halos, 3), generator=g)
    lone = torch.rand(halos, generator=g) < 0.6
    pos = torch.where(lone[:, None], torch.rand((halos, 3), generator=g) * box, pos)
    rec = torch.randn((halos, nf), generator=g)
    rec[:, 0:3] = pos - 0.5 * box
    rec[:, 3:6] *= 5.0
    rec[:, 6] = torch.clamp(3.0 * torch.exp(0.45 * torch.randn(halos, generator=g)), 1.0, 30.0)
    rec[:, 7:10] *= 0.3
    return rec.to(DEV)


def prepare(case, seed):
    op = case["op"]
    s = dict(case=case)
    if op in ("shell", "tiles"):
        ct = read_homeltab(WEBSKY_TABLE)
        s.update(ct=ct, fcrit=api.fsc_of_z(ct, 0.0), tables=api.build_shell_tables(case["nhunt"]))
        if op == "shell":
            s["tile"] = _tile(case["n"], case["nbuff"], _radii(case), case["peaks"], seed)
        else:
            sides = [int(n) for n in case["sides"].split()]
            s["tiles"] = [_tile(n, case["nbuff"], _radii(case),
                                _cap(n, case["nbuff"], case["nfilt"]), 1000 * seed + q)
                          for q, n in enumerate(sides)]
    elif op in ("peaks", "bank"):
        n = case["n"]
        fields, dk = synth.fields_torch(n, n * ALATT, seed, DEV, second_order=False)
        s["mask"] = api.to_device_field(torch.zeros((n, n, n), dtype=torch.int8, device=DEV),
                                        dtype=torch.int8)
        s["radii"] = _radii(case)
        s["fcrit"] = [1.5] * case["nfilt"]
        s["capacity"] = case["peaks"]
        if op == "peaks":
            s["smoothed"] = [api.to_device_field(synth.smooth_tophat_torch(dk, n, n * ALATT, R))
                             for R in s["radii"]]
        else:
            s["delta"] = api.to_device_field(fields["delta"])
    elif op == "convolve":
        n_in = case["n"] + 2 * case["nshell"]
        s["pk"] = synth.PowerSpectrum()
        s["noise"] = api.to_device_field(_noise(n_in, seed))
    elif op == "lpt":
        n = case["n"]
        s["delta"] = api.to_device_field(
            synth.fields_torch(n, n * ALATT, seed, DEV, second_order=False)[0]["delta"])
    elif op == "coarse":
        s["coarse"] = [api.to_device_field(v) for v in _coarse_inputs(case, seed)]
        s["seed"] = seed
    else:
        cos = cosmology.CosmologyParams(0.31, 0.049, 0.69, 0.68)
        rec = _records(case["halos"], case["nf"], seed)
        # the program's catalog arrays: merge and finalisation give a varying number of halos
        s.update(records=rec, merged=torch.zeros_like(rec), final=torch.zeros_like(rec), cos=cos,
                 growth=cosmology.dlinear_tables(cos),
                 chi2z=cosmology.build_chi_to_z(cos, z_max=10.0))
    return s


def _noise(n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn((n, n, n), generator=g, device=DEV)


def _coarse_inputs(case, seed):
    """The coarse white noise and four large-scale fields (delta, psi_1) on the M^3 grid."""
    M, out = case["M"], []
    for q in range(5):
        out.append(_noise(M, 5 * seed + q))
    return out


# ---------------------------------------------------------------- one pass

def run(s):
    c = s["case"]
    op = c["op"]
    if op == "shell":
        t = s["tile"]
        t["mask"].zero_()
        r = api.shell_analyse(t["fields"], t["pi"], t["pj"], t["pk"], t["Rf"], t["ir2min"],
                              s["tables"], s["ct"], alatt=ALATT, ZZon=1.0, fcrit=s["fcrit"],
                              nbuff=c["nbuff"], variant=c["variant"], mask=t["mask"])
        return {"results": r, "mask": t["mask"]}
    if op == "tiles":
        for t in s["tiles"]:
            t["mask"].zero_()
        r = api.shell_analyse_tiles(s["tiles"], s["tables"], s["ct"], alatt=ALATT, ZZon=1.0,
                                    fcrit=s["fcrit"], nbuff=c["nbuff"], variant=c["variant"])
        # one catalog of the batch
        return {"results": {k: torch.cat([x[k] for x in r]) for k in r[0]},
                "masks": [t["mask"] for t in s["tiles"]]}
    if op == "peaks":
        s["mask"].zero_()
        pk = api.peak_find(s["smoothed"], s["fcrit"], c["nbuff"], s["mask"],
                           capacity=s["capacity"])
        return {"peaks": pk, "mask": s["mask"]}
    if op == "bank":
        s["mask"].zero_()
        pk = api.peak_find_tile(s["delta"], s["radii"], s["fcrit"], c["nbuff"], s["mask"],
                                alatt=ALATT, wsmooth=c["wsmooth"], with_lapd=c["lapd"],
                                capacity=s["capacity"])
        return {"peaks": pk, "mask": s["mask"]}
    if op == "convolve":
        return api.isolated_convolve_gpu_multi(
            s["noise"], s["pk"].file, c["n"] * ALATT, c["n"],
            kernels=[(0, 0, 0), (1, 1, 0), (1, 2, 0), (1, 3, 0)], nshell=c["nshell"],
            return_device=True)
    if op == "lpt":
        n = c["n"]
        psi2 = api.compute_2lpt_gpu(s["delta"], n, n * ALATT, return_device=True)
        return list(psi2) + [api.compute_laplacian_gpu(s["delta"], n, n * ALATT,
                                                       return_device=True)]
    if op == "coarse":
        N, t = c["block"] * c["M"], c["tile"]
        res = api.generate_extended_residual(t, t, t, c["nsub"], c["nmesh"], N, s["seed"],
                                             s["coarse"][0], c["M"], 0, return_device=True)
        return [res] + [api.interpolate_to_tile_gpu(f, t, t, t, c["nsub"], c["nmesh"], N,
                                                    c["M"], return_device=True)
                        for f in s["coarse"][1:]]
    merged = api.merge_catalog(s["records"], volume_reduction=True)
    k = len(merged)
    s["merged"][:k] = merged
    s["merged"][k:] = 0.0
    api.finalize_eulerian(merged, s["growth"], OBS, Om=s["cos"].Om, OL=s["cos"].OL, ievol=1,
                          chi2z=s["chi2z"], out=s["final"][:k])
    s["final"][k:] = 0.0
    return {"merged": s["merged"], "final": s["final"]}


# ---------------------------------------------------------------- work of one pass

def work(case):
    op = case["op"]
    if op in ("shell", "tiles"):
        sides = [case["n"]] if op == "shell" else [int(v) for v in case["sides"].split()]
        b = f = 0.0
        for n in sides:
            np_ = case.get("peaks") or _cap(n, case["nbuff"], case["nfilt"])
            # 7 fields once, the mask written, 24 B in and 284 B out per peak
            b += 7.0 * 4 * n ** 3 + (n - 2 * case["nbuff"]) ** 3 + 308.0 * np_
            # about 600 cells per peak to the shell its results need: 22 sums, 15 products
            f += 600.0 * 37.0 * np_
        return {"bytes": b, "flops": f}
    if op == "peaks":
        m3 = (case["n"] - 2 * case["nbuff"]) ** 3
        return {"bytes": 4.0 * case["nfilt"] * m3 + m3 + 20.0 * case["peaks"],
                "flops": 27.0 * case["nfilt"] * m3}
    if op == "bank":
        n, k = case["n"], case["nfilt"] * (2 if case["lapd"] else 1)
        m3 = (n - 2 * case["nbuff"]) ** 3
        fft = 2.5 * n ** 3 * math.log2(n ** 3)
        return {"bytes": 4.0 * n ** 3 + m3 + 20.0 * case["peaks"], "flops": fft * (1 + k)}
    if op == "convolve":
        n, L = case["n"], 2 * (case["n"] + 2 * case["nshell"])
        return {"bytes": 4.0 * (L // 2) ** 3 + 16.0 * n ** 3,
                "flops": 5 * 2.5 * L ** 3 * math.log2(L ** 3)}
    if op == "lpt":
        n = case["n"]
        return {"bytes": 20.0 * n ** 3, "flops": 13 * 2.5 * n ** 3 * math.log2(n ** 3)}
    if op == "coarse":
        n3 = case["nmesh"] ** 3
        # 60 integer and 40 float operations a Gaussian; 128 a tri-cubic cell
        return {"bytes": 20.0 * n3 + 20.0 * case["M"] ** 3, "flops": (100.0 + 4 * 128.0) * n3}
    N = case["halos"]
    # the records in, the two catalogs out
    return {"bytes": 4.0 * case["nf"] * N * 3, "flops": 600.0 * N}


# ---------------------------------------------------------------- 64-bit values

def exact(case, seed):
    op = case["op"]
    if op == "convolve":
        return _exact_convolve(case, seed)
    if op == "lpt":
        return _exact_lpt(case, seed)
    if op == "coarse":
        return _exact_coarse(case, seed)
    if op == "catalog" and case["halos"] <= 6000:
        return _exact_catalog(case, seed)
    if op == "shell" and case["n"] <= 44 and case["variant"] == "C" and case["nfilt"] <= 8:
        return _exact_shell(case, seed)
    # peak lists are choices among the smoothed values, so their entries have no 64-bit
    # counterpart at the same place; larger tiles and catalogs take minutes here
    return None


def _freq(n, box, nyq_sign=-1.0):
    dk = 2.0 * math.pi / box
    kx = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float64)
    f = torch.fft.fftfreq(n, d=1.0 / n, device=DEV, dtype=torch.float64)
    if n % 2 == 0:
        f = torch.where(f == -(n // 2), nyq_sign * (n // 2), f)
    return kx[None, None, :] * dk, f[None, :, None] * dk, f[:, None, None] * dk


def _exact_convolve(case, seed):
    n, ns = case["n"], case["nshell"]
    n_in = n + 2 * ns
    L = 2 * n_in
    noise = _noise(n_in, seed).permute(2, 1, 0).double()  # [k, j, i]
    spec = torch.fft.rfftn(noise, s=(L, L, L))
    box = L * ALATT
    KX, KY, KZ = _freq(L, box)
    dk = 2.0 * math.pi / box
    # sqrt P(k) as the method tabulates it: 8192 points uniform in ln k, linear between them
    lk = np.linspace(math.log(dk * 0.5), math.log(math.sqrt(3.0) * (L / 2) * dk * 1.5), 8192)
    tab = np.sqrt(synth.PowerSpectrum().file(np.exp(lk)) * dk ** 3 * float(L) ** 3)
    tab = torch.as_tensor(tab, device=DEV)
    out = []
    for kind, d in ((0, 0), (1, 1), (1, 2), (1, 3)):
        w = spec.clone()
        for z0 in range(0, L, 64):
            sl = slice(z0, min(L, z0 + 64))
            k2 = KX ** 2 + KY ** 2 + KZ[sl] ** 2
            zero = k2 == 0
            k2 = torch.where(zero, torch.ones_like(k2), k2)
            pos = (0.5 * torch.log(k2) - lk[0]) / (lk[1] - lk[0])
            i0 = torch.clamp(torch.floor(pos), 0, len(lk) - 2).long()
            amp = tab[i0] + torch.clamp(pos - i0, 0.0, 1.0) * (tab[i0 + 1] - tab[i0])
            amp = torch.where(zero, torch.zeros_like(amp), amp)
            if kind == 0:
                w[sl] *= amp
            else:
                comp = (KX, KY, KZ[sl])[d - 1]
                w[sl] *= 1j * comp * amp / k2
        # the inverse real transform of the planes made Hermitian
        for p in (0, L // 2):
            a = w[:, :, p]
            b = torch.roll(torch.flip(a, (0, 1)), (1, 1), (0, 1)).conj()
            w[:, :, p] = 0.5 * (a + b)
        f = torch.fft.irfftn(w, s=(L, L, L))
        out.append(f[ns:ns + n, ns:ns + n, ns:ns + n].permute(2, 1, 0).contiguous())
        del w, f
    return out


def _exact_lpt(case, seed):
    n = case["n"]
    box = n * ALATT
    d = synth.fields_torch(n, box, seed, DEV, second_order=False)[0]["delta"]
    d = d.permute(2, 1, 0).double()
    spec = torch.fft.rfftn(d)
    KX, KY, KZ = _freq(n, box, nyq_sign=1.0)
    K = (KX, KY, KZ)
    k2 = KX ** 2 + KY ** 2 + KZ ** 2
    inv = torch.where(k2 > 0, 1.0 / torch.where(k2 > 0, k2, torch.ones_like(k2)),
                      torch.zeros_like(k2))
    src = 0.5 * d * d
    for a in range(3):
        for b in range(a, 3):
            phi = torch.fft.irfftn(-K[a] * K[b] * inv * spec, s=(n, n, n))
            src -= phi * phi * (0.5 if a == b else 1.0)
            del phi
    half = n // 2
    ix = torch.arange(half + 1, device=DEV)[None, None, :]
    iy = torch.arange(n, device=DEV)
    keep = ~((ix == half) | (iy[None, :, None] == half) | (iy[:, None, None] == half))
    sk = torch.fft.rfftn(src)
    del src
    out = [torch.fft.irfftn(-1j * K[a] * inv * sk * keep, s=(n, n, n)) for a in range(3)]
    out.append(torch.fft.irfftn(k2 * spec * keep, s=(n, n, n)))
    return [o.permute(2, 1, 0) for o in out]


def _threefry_gauss(idx, seed):
    """Gaussian of global cell idx (int64 tensor): Threefry-2x64-20 of counter (idx >> 1, 0)
    under key (seed, 0), Box-Muller, the cosine for an even cell and the sine for an odd one."""
    rot = (16, 42, 12, 31, 16, 32, 24, 21)
    par = 0x1BD11BDAA9FC1A22 ^ seed
    ks = (seed, 0, par)

    def rotl(x, r):
        return (x << r) | ((x >> (64 - r)) & ((1 << r) - 1))

    x0 = (idx >> 1) + ks[0]
    x1 = torch.zeros_like(idx)
    for r in range(20):
        x0 = x0 + x1
        x1 = rotl(x1, rot[r % 8]) ^ x0
        if r % 4 == 3:
            q = (r + 1) // 4
            x0 = x0 + ks[q % 3]
            x1 = x1 + ks[(q + 1) % 3] + q

    def unit(x):
        return (((x >> 11) & ((1 << 53) - 1)).double() + 1.0) * 2.0 ** -53

    th = 2.0 * math.pi * unit(x1)
    return torch.sqrt(-2.0 * torch.log(unit(x0))) * torch.where(idx & 1 == 1, torch.sin(th),
                                                               torch.cos(th))


def _exact_coarse(case, seed):
    nm, M, B, t = case["nmesh"], case["M"], case["block"], case["tile"]
    N = M * B
    start = (t - 1) * case["nsub"] - (nm - case["nsub"]) // 2  # 0-based
    g = torch.remainder(torch.arange(start, start + nm, device=DEV), N)
    cs = [v.permute(2, 1, 0).double() for v in _coarse_inputs(case, seed)]  # [k, j, i]
    b = g // B
    mean = cs[0][b][:, b][:, :, b] / math.sqrt(float(B) ** 3)
    fine = torch.empty((nm, nm, nm), dtype=torch.float64, device=DEV)
    for z in range(nm):
        idx = g[None, :] + g[:, None] * N + g[z] * N * N
        fine[z] = _threefry_gauss(idx, seed)
    out = [(fine - mean).permute(2, 1, 0)]
    # Catmull-Rom, cell-centred on both grids, the same along each axis
    f = (g.double() + 0.5) / B + 0.5
    i0 = torch.floor(f)
    u = f - i0
    w = (-0.5 * u ** 3 + u ** 2 - 0.5 * u, 1.5 * u ** 3 - 2.5 * u ** 2 + 1.0,
         -1.5 * u ** 3 + 2.0 * u ** 2 + 0.5 * u, 0.5 * u ** 3 - 0.5 * u ** 2)
    A = torch.zeros((nm, M), dtype=torch.float64, device=DEV)
    for q in range(4):
        A.scatter_add_(1, torch.remainder(i0.long() - 2 + q, M)[:, None], w[q][:, None])
    for v in cs[1:]:
        v = torch.tensordot(A, v, dims=([1], [0]))
        v = torch.tensordot(v, A, dims=([1], [1])).permute(0, 2, 1)
        v = torch.tensordot(v, A, dims=([2], [1]))
        out.append(v.permute(2, 1, 0))
    return out


def _exact_catalog(case, seed):
    rec = _records(case["halos"], case["nf"], seed)
    x, r = rec[:, 0:3].double(), rec[:, 6].double()
    N = len(r)
    cpu = rec.cpu().numpy()
    order = np.lexsort((cpu[:, 2], cpu[:, 1], cpu[:, 0], -cpu[:, 6]))
    rank = torch.empty(N, dtype=torch.long, device=DEV)
    rank[torch.as_tensor(order, device=DEV)] = torch.arange(N, device=DEV)
    d = torch.sqrt(((x[:, None, :] - x[None, :, :]) ** 2).sum(-1))
    lower = rank[:, None] < rank[None, :]
    holds = ((d < r[:, None]) & lower).cpu().numpy()
    alive = np.ones(N, bool)
    for p in order:
        if alive[p]:
            alive &= ~holds[p]
    live = torch.as_tensor(alive, device=DEV)
    r1, r2 = r[:, None], r[None, :]
    cut = lower & live[:, None] & live[None, :] & (d < r1 + r2) & (d > (r1 - r2).abs())
    dd = torch.where(d > 0, d, torch.ones_like(d))
    h1 = (r2 - r1 + d) * (r2 + r1 - d) / (2.0 * dd)
    h2 = (r1 - r2 + d) * (r1 + r2 - d) / (2.0 * dd)
    v1 = torch.where(cut, math.pi / 3.0 * h1 ** 2 * (3.0 * r1 - h1), torch.zeros_like(d))
    v2 = torch.where(cut, math.pi / 3.0 * h2 ** 2 * (3.0 * r2 - h2), torch.zeros_like(d))
    vol = 4.0 * math.pi / 3.0 * r ** 3 - v1.sum(1) - v2.sum(0)
    keep = live & (vol > 0)
    merged = torch.zeros((N, case["nf"]), dtype=torch.float64, device=DEV)
    k = int(keep.sum())
    merged[:k] = rec.double()[keep]
    merged[:k, 6] = (vol[keep] * 3.0 / (4.0 * math.pi)) ** (1.0 / 3.0)
    # Eulerian positions and velocities at the redshift of each halo's distance
    fin = merged[:k].cpu().numpy()
    cos = cosmology.CosmologyParams(0.31, 0.049, 0.69, 0.68)
    at, _, ft = (np.asarray(v) for v in cosmology.dlinear_tables(cos))
    zs, chis, _ = cosmology.build_chi_to_z(cos, z_max=10.0)
    d1, d2 = fin[:, 3:6].copy(), fin[:, 7:10].copy()
    fin[:, 0:3] += d1 + d2
    a = 1.0 / (1.0 + np.interp(np.sqrt(((fin[:, 0:3] - np.array(OBS)) ** 2).sum(1)), chis, zs))
    q = np.clip(np.searchsorted(at, a) - 2, 0, len(at) - 4)  # four growth-table points about a
    f = np.zeros(k)
    for u in range(4):
        w = ft[q + u].copy()
        for v in range(4):
            if v != u:
                w *= (a - at[q + v]) / (at[q + u] - at[q + v])
        f += w
    fin[:, 3:6] = (a * 100.0 * np.sqrt(cos.Om * a ** -3.0 + cos.OL) * f)[:, None] * (d1 + 2 * d2)
    fin[:, 7:10] = 0.0
    final = torch.zeros_like(merged)
    final[:k] = torch.as_tensor(fin, device=DEV)
    return {"merged": merged, "final": final}


def _exact_shell(case, seed):
    """Every candidate of a small tile in numpy: sums over all shells of the hunt radius, the
    crossing of fcrit, the inward walk to the collapse, the record fields."""
    t = _tile(case["n"], case["nbuff"], _radii(case), case["peaks"], seed)
    ct = read_homeltab(WEBSKY_TABLE)
    fcrit = api.fsc_of_z(ct, 0.0)
    f = {k: v.cpu().numpy().astype(np.float64) for k, v in t["fields"].items()}
    f["deltaT"] = np.transpose(f["delta"], (1, 2, 0))  # [i, j, k] -> delta[k, i, j]
    n, R = case["n"], case["nhunt"]
    a = np.arange(-R, R + 1)
    off = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    r2 = (off ** 2).sum(1)
    off, r2 = off[r2 <= R * R], r2[r2 <= R * R]
    u2 = np.unique(r2)
    sh = np.searchsorted(u2, r2)  # 0-based shell of each offset
    NS = len(u2)
    rad = np.concatenate([[0.0], np.sqrt(u2), [0.0]])  # 1-based
    m = NS - 1
    wR, aR = 3.0 / (4.0 * math.pi) / ALATT, 3.0 / ALATT
    tab = np.asarray(ct["table"], np.float64)

    def hR(u0, u12):
        x = abs(u0)
        if x >= 2.0:
            return 0.0
        v = 1.6 * u12 - 6.4 / 7.0
        if x >= 1.0:
            return (v - x ** 2 * (4 - x * (4 - x * (1.5 - 0.2 * x))) * u12
                    + x ** 4 * (2 - x * (2.4 - x * (1 - x / 7.0))))
        v -= 0.2 * (u12 - 1.0 / 7.0)
        return (v - x ** 2 * (2 - x ** 2 * (1.5 - 0.6 * x)) * u12
                + x ** 4 * (1 - x ** 2 * (1 - 3 * x / 7.0)))

    W = np.zeros((NS + 2, NS + 2))
    for p in range(2, NS + 1):
        for q in range(2, NS + 1):
            d0, d1 = rad[p] - rad[q], rad[p] ** 2 + rad[q] ** 2
            if d0 * d0 < 4.0:
                W[p, q] = hR(d0, d1) / (d1 - d0 * d0) ** 2

    def akk(u):
        ru = math.sqrt(u)
        if ru < 1.0:
            return 3.0 / (2.0 * math.pi) * (2.0 / 3.0 - u + 0.5 * u * ru)
        return (2.0 - ru) ** 3 / (4.0 * math.pi) if ru <= 2.0 else 0.0

    def strain(X, p, lo, hi):
        """X [shell, 12] (gradients, transposed gradients, symmetric strain) -> E33, g, gf"""
        v = np.zeros(12)
        if p > 1:
            for q in range(lo, hi + 1):
                v += W[p, q] * X[q]
            v *= wR / rad[p]
        else:
            for q in range(lo, hi + 1):
                con = 100.0 * rad[q] ** 2
                if con < 1100.0:
                    i = int(con)
                    y = akk(0.01 * i) + (con - i) * (akk(0.01 * (i + 1)) - akk(0.01 * i))
                    v += (0.5 * y / rad[q] if rad[q] > 0 else math.inf) * X[q]
            v *= aR
        e = -0.5 * v[6:]
        return np.array([[e[0], e[1], e[2]], [e[1], e[3], e[4]], [e[2], e[4], e[5]]]), v[:6]

    def ev(E):
        lam = np.linalg.eigvalsh(E) if np.isfinite(E).all() else np.full(3, np.nan)
        F = lam.sum()
        if not F > 0:
            return lam, F, 0.0, 0.0
        return lam, F, 0.5 * (lam[2] - lam[0]) / F, 0.5 * (lam[2] + lam[0] - 2 * lam[1]) / F

    def zvir(Fb, e, p):
        if not Fb > 0:
            return -1.0
        q = (math.log10(Fb), e, 0.0 if e < 1e-5 else p / e)
        idx, w = [], []
        for x, lo, hi, c in zip(q, (ct["x1"], ct["y1"], ct["z1"]), (ct["x2"], ct["y2"], ct["z2"]),
                                tab.shape):
            if not lo <= x <= hi:
                return -1.0
            g = (x - lo) / ((hi - lo) / (c - 1))
            i = min(max(int(math.floor(g)), 0), c - 2)
            idx.append(i)
            w.append(g - i)
        v = 0.0
        for bx in (0, 1):
            for by in (0, 1):
                for bz in (0, 1):
                    v += (tab[idx[0] + bx, idx[1] + by, idx[2] + bz]
                          * (w[0] if bx else 1 - w[0]) * (w[1] if by else 1 - w[1])
                          * (w[2] if bz else 1 - w[2]))
        return v

    def first(lo, hi, ok):
        for q in range(lo, hi + 1):
            if ok(q):
                return q
        return hi + 1

    npk = len(t["pi"])
    out = {k: np.zeros(npk) for k in ("RTHL", "Fbarx", "e_v", "p_v", "Srb", "d2F", "zvir_half")}
    out.update({k: np.zeros((npk, 3)) for k in ("eigs", "Sbar", "Sbar2", "gradpk", "gradpkf",
                                                "gradpkrf")})
    out["strain"] = np.zeros((npk, 3, 3))
    out["RTHL"][:] = out["zvir_half"][:] = -1.0
    peaks = torch.stack([t["pi"], t["pj"], t["pk"]], 1).cpu().numpy() - 1
    Rfs, irs = t["Rf"].cpu().numpy(), t["ir2min"].cpu().numpy()
    with np.errstate(all="ignore"):
        for p in range(npk):
            cell = peaks[p] + off
            ok = ((cell >= 0) & (cell < n)).all(1)
            i, j, k = cell[ok].T
            o, s = off[ok].astype(np.float64), sh[ok]

            def sums(v):
                return np.bincount(s, v, NS)

            cnt = sums(np.ones(len(s)))
            de, dt = f["delta"][i, j, k], f["deltaT"][i, j, k]
            ps = [f[key][i, j, k] for key in ("etax", "etay", "etaz")]
            p2 = [f[key][i, j, k] for key in ("eta2x", "eta2y", "eta2z")]
            X = np.zeros((NS + 2, 12))
            rr = rad[1:NS + 1]
            SR = [[sums(ps[L] * o[:, K]) / rr for K in range(3)] for L in range(3)]
            for K in range(3):
                X[2:NS + 1, K] = (sums(de * o[:, K]) / rr)[1:]
                X[2:NS + 1, 3 + K] = (sums(dt * o[:, K]) / rr)[1:]
            for q, (L, K) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
                X[2:NS + 1, 6 + q] = (SR[L][K] + SR[K][L])[1:]
            F = sums(de)
            Fb = np.zeros(NS + 2)
            Fb[1] = prev = F[0]
            for q in range(2, NS + 1):
                dF = F[q - 1] / cnt[q - 1] if cnt[q - 1] > 0 else 0.0
                Fb[q] = (rad[q - 1] ** 3 * Fb[q - 1] + 0.5 * (prev + dF)
                         * (rad[q] ** 3 - rad[q - 1] ** 3)) / rad[q] ** 3
                prev = dF
            # filter-scale gradient
            rf2 = (Rfs[p] / ALATT) ** 2
            dist = np.abs(u2[1:m] - rf2)
            mrf = int(np.argmin(dist)) + 1 if dist.min() < 10.0 else 1
            lo = first(1, mrf - 1, lambda q: rad[q] > max(rad[mrf] - 2.0, 0.0))
            hi = first(mrf + 1, m, lambda q: rad[q] >= rad[mrf] + 2.0) - 1
            grf = strain(X, mrf, min(lo, mrf), hi)[1]
            # crossing
            m0 = min(first(2, m, lambda q: u2[q - 1] > irs[p]), m)
            mupp = None
            if Fb[m0] >= fcrit:
                q = first(m0, m, lambda q: Fb[q] < fcrit)
                if q <= m:
                    m0 = q
                else:
                    mupp = m
            else:
                found = False
                for q in range(max(m0 - 1, 1), 0, -1):
                    if Fb[q] >= fcrit:
                        found = True
                        break
                    m0 = q
                if not found:
                    continue
            if mupp is None:
                mupp = first(m0 + 1, m, lambda q: rad[q] >= rad[m0] + 2.0) - 1
            mlow = min(first(1, m0 - 1, lambda q: rad[q] > max(rad[m0] - 2.0, 0.0)), m0)
            if m0 == 1:
                continue
            E, g = strain(X, m0, mlow, mupp)
            Frhoh = ev(E)[1]
            last, before = (E, g), (E, g)
            z1, hit = -1.0, False
            for q in range(m0 - 1, 0, -1):
                up, dn = rad[q] + 2.0, max(rad[q] - 2.0, 0.0)
                if rad[mupp] > up:
                    mupp = max([q] + [v for v in range(q + 1, mupp + 1) if rad[v] < up])
                if mlow > 1 and rad[mlow - 1] > dn:
                    mlow = min([mlow] + [v for v in range(mlow - 1, 0, -1) if rad[v] > dn])
                cur = strain(X, q, mlow, mupp)
                lam, Fr, e, pv = ev(cur[0])
                z = zvir(Fb[q], e, pv)
                last, Frhoh = cur, Fr
                if z >= 1.0:
                    m0, zp, hit = q + 1, z, True
                    break
                z1, before = z, cur
            if not hit:
                continue
            ra, rb = rad[m0 - 1] ** 3, rad[m0] ** 3
            dz = zp - z1
            r3 = ra + (rb - ra) * (zp - 1.0) / dz if z1 > 0 and dz != 0 else ra
            RT = r3 ** (1.0 / 3.0)
            if RT <= 0:
                continue
            if z1 > 0 and rb != ra:
                w = (r3 - ra) / (rb - ra)
                Fx = Fb[m0 - 1] + w * (Fb[m0] - Fb[m0 - 1])
                E = last[0] + w * (before[0] - last[0])
                g = last[1] + w * (before[1] - last[1])
            else:
                Fx, E, g = Fb[m0 - 1], last[0], before[1]
            tr = np.trace(E)
            lam, _, e, pv = ev(E * (Fx / tr) if tr != 0 else E)
            inner = s <= m0 - 2
            nin = inner.sum()
            srb, r5 = 0.0, 0.0
            for q in range(2, m0):
                srb += 0.5 * (Fb[q - 1] + Fb[q]) * (rad[q] ** 5 - r5)
                r5 = rad[q] ** 5
            if z1 > 0 and dz != 0:
                srb += 0.5 * (Fb[m0 - 1] + Fx) * (RT ** 5 - r5)
            if Fx * RT ** 5 > 0:
                srb /= Fx * RT ** 5
            zh = -1.0
            if RT >= 3.0:
                for q in range(10):
                    rc = RT * (q / 9.0 * 0.5 + 0.5) ** (1.0 / 3.0)
                    hi = min(first(2, m - 1, lambda v: rad[v] > rc + 2.0), m - 1)
                    lo = first(1, m - 1, lambda v: rad[v] > max(rc - 2.0, 0.0))
                    c0 = min(first(1, m - 1, lambda v: rad[v] > rc), m - 1)
                    _, _, ee, pp = ev(strain(X, c0, lo if lo <= m - 1 else 1, hi)[0])
                    zh = max(zh, zvir(Fb[c0], ee, pp) - 1.0)
            out["RTHL"][p], out["Fbarx"][p], out["e_v"][p], out["p_v"][p] = RT, Fx, e, pv
            out["Srb"][p], out["zvir_half"][p] = srb, zh
            out["strain"][p] = last[0] * (Fx / Frhoh) if Frhoh != 0 else last[0]
            out["eigs"][p], out["gradpk"][p], out["gradpkf"][p] = lam, g[:3], g[3:]
            out["gradpkrf"][p] = grf[:3]
            out["Sbar"][p] = [v[inner].sum() / nin for v in ps]
            out["Sbar2"][p] = [v[inner].sum() / nin for v in p2]
    res = {k: torch.as_tensor(v) for k, v in out.items()}
    res.update({k: None for k in ("nshells_used", "crossing_shell", "bracket")})
    return {"results": res, "mask": None}
