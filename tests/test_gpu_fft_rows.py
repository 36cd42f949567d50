"""The row passes of short transforms (8 to 64 points: a thread per element instead of a wavefront per
piece of 64) and the 128-point ones beside them, whole, padded and cropped with odd starts and
sides, against the oracle: relative L2 <= 5e-6 for the isolated convolution, 1e-5 for the periodic
fields, the bars of the tests of those entries at larger sizes."""
import numpy as np
import pytest

from huntian_hip import api
from oracle import fields as F

pytestmark = pytest.mark.gpu


def pk_test(k):
    return 100.0 / (1.0 + (np.asarray(k) * 50.0) ** 4)


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n_input,nshell", [(4, 0), (4, 1), (8, 3), (16, 0), (16, 5), (32, 1), (64, 3)])
def test_isolated(n_input, nshell):
    rng = np.random.default_rng(n_input + nshell)
    n, box = n_input - 2 * nshell, 100.0
    noise = rng.standard_normal((n_input,) * 3).astype(np.float32)
    kernels = [(0, 0, 0), (1, 2, 0), (2, 1, 3)]
    got = api.isolated_convolve_gpu_multi(noise, pk_test, box, n, kernels=kernels, nshell=nshell)
    for kern, g in zip(kernels, got):
        assert rel(g, F.isolated_convolve(noise, pk_test, box, n, kern, nshell=nshell)) <= 5e-6, kern


@pytest.mark.parametrize("n", [8, 16, 32, 64, 128])
def test_periodic(n):
    rng = np.random.default_rng(n)
    # smooth enough that the second-order source is not a difference of large terms
    spec = np.fft.rfftn(rng.standard_normal((n,) * 3))
    k = np.fft.fftfreq(n, 1.0 / n)
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + np.arange(n // 2 + 1)[None, None, :] ** 2
    delta = np.fft.irfftn(spec * np.exp(-k2 / (n / 6.0) ** 2), s=(n,) * 3, axes=(0, 1, 2)).astype(np.float32)
    for g, w in zip(api.compute_2lpt_gpu(delta, n, 2.0 * n), F.compute_2lpt(delta, n, 2.0 * n)):
        assert rel(g, w) <= 1e-5
    assert rel(api.compute_laplacian_gpu(delta, n, 2.0 * n), F.compute_laplacian(delta, n, 2.0 * n)) <= 1e-5
