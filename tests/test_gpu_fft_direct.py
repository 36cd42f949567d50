"""The 128- to 512-point column passes and the 512-point rows with the spectrum loaded straight
into LDS (tuning fft_direct = 1) and through registers (0): the same bits for padded and cropped
transforms, crops of odd start and side (single reals stored instead of pairs) included, and
against the oracle to the tolerance of the isolated convolutions (relative L2 <= 5e-6)."""
import numpy as np
import pytest

from huntian_hip import api
from oracle import fields as F

pytestmark = pytest.mark.gpu


def pk_test(k):
    return 100.0 / (1.0 + (np.asarray(k) * 50.0) ** 4)


@pytest.mark.parametrize("n_input,nshell", [(64, 0), (64, 3), (128, 5), (128, 20), (256, 0), (256, 1)])
def test_direct_columns_and_rows(n_input, nshell):
    import torch

    ctx = api.context(0)
    rng = np.random.default_rng(n_input + nshell)
    n, box = n_input - 2 * nshell, 100.0
    noise = rng.standard_normal((n_input,) * 3).astype(np.float32)
    delta = rng.standard_normal((n_input,) * 3).astype(np.float32)
    kernels = [(0, 0, 0), (1, 2, 0)]
    out = {}
    try:
        for direct in (1, 0):
            ctx.set_tuning(fft_direct=direct)
            conv = api.isolated_convolve_gpu_multi(noise, pk_test, box, n, kernels=kernels,
                                                   nshell=nshell, return_device=True)
            psi = api.compute_2lpt_gpu(delta, n_input, box, return_device=True)
            out[direct] = list(conv) + list(psi)
            print("direct", direct, n_input, nshell, flush=True)
    finally:
        ctx.set_tuning(fft_direct=1)
    for a, b in zip(out[1], out[0]):
        assert torch.equal(a, b)
    if n_input <= 128:
        for kern, got in zip(kernels, out[1]):
            ref = F.isolated_convolve(noise, pk_test, box, n, kern, nshell=nshell)
            g = got.cpu().numpy().astype(np.float64)
            assert np.linalg.norm(g - ref) / np.linalg.norm(ref) <= 5e-6
