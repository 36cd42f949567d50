"""Fields and outputs that start 4 bytes past an aligned address, which the wider loads and stores
leave to their 4-byte forms: the same bits as from aligned ones."""
import numpy as np
import pytest
import torch

from huntian_hip import api, synth
from test_gpu_shell_blocks import _fields, _peaks, _same

pytestmark = pytest.mark.gpu


def _shift(t):
    """The same column-major field at an address 4 bytes past a 16-byte line."""
    n = t.shape[0]
    out = torch.empty(n ** 3 + 1, device=t.device)[1:].view(n, n, n).permute(2, 1, 0)
    out.copy_(t)
    assert out.data_ptr() % 8 == 4
    return out


def _shifted_out(n, dev, k=1):
    return [torch.empty(n ** 3 + 1, device=dev)[1:].view(n, n, n).permute(2, 1, 0) for _ in range(k)]


@pytest.mark.parametrize("n,nshell", [(16, 0), (64, 2), (128, 0), (256, 0), (512, 0)])
def test_transforms(monkeypatch, n, nshell):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = api.to_device_field(torch.randn((n,) * 3, generator=g, device="cuda"))
    pk = synth.PowerSpectrum().file

    def run(f):
        out = []
        if n <= 256:
            m = n - 2 * nshell
            out += api.isolated_convolve_gpu_multi(f, pk, 2.0 * m, m, kernels=[(0, 0, 0), (1, 2, 0)],
                                                   nshell=nshell, return_device=True)
        out += api.compute_2lpt_gpu(f, n, 2.0 * n, return_device=True)
        out.append(api.compute_laplacian_gpu(f, n, 2.0 * n, return_device=True))
        print("transforms", n, f.data_ptr() % 16, flush=True)
        return out

    want = run(x)
    shifted_in = run(_shift(x))
    monkeypatch.setattr(api, "_field_out", _shifted_out)
    for a, b, c in zip(want, shifted_in, run(_shift(x))):
        assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("which", ["delta", "etay", "all"])
def test_shell_analysis(websky, which):
    n, nhunt = 64, 12
    f, pk = _fields(n, 21, True), _peaks(n, 4000, 22)
    shifted = {k: _shift(v) if which in (k, "all") else v for k, v in f.items()}
    kw = dict(alatt=2.0, ZZon=1.0, fcrit=api.fsc_of_z(websky, 0.0))
    arg = (pk["pi"], pk["pj"], pk["pk"], pk["Rf"], pk["ir2min"], api.build_shell_tables(nhunt), websky)
    _same(api.shell_analyse(shifted, *arg, **kw), api.shell_analyse(f, *arg, **kw), which)


def test_peak_finding():
    n = 96
    g = torch.Generator(device="cuda").manual_seed(3)
    sm = [api.to_device_field(torch.randn((n,) * 3, generator=g, device="cuda")) for _ in range(3)]

    def run(fields):
        mask = api.fortran_empty((n, n, n), torch.int8)
        mask.zero_()
        r = api.peak_find(fields, [1.0] * 3, 5, mask, capacity=n ** 3 // 8)
        b = api.peak_find_tile(fields[0], [6.0, 3.0], [0.1] * 2, 4, mask, alatt=2.0, with_lapd=True)
        return r, b, mask

    a, b = run(sm), run([_shift(f) for f in sm])
    assert a[0]["total"] == b[0]["total"] > 1000 and a[1]["total"] == b[1]["total"] > 100
    for x, y in zip(a[:2], b[:2]):
        for k in ("i", "j", "k", "filt", "delta"):
            assert np.array_equal(x[k].cpu().numpy(), y[k].cpu().numpy()), k
    assert torch.equal(a[2], b[2])
