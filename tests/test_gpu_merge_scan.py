"""The neighbour scans of hnt_merge_catalog where their lists run over: more containment edges or
overlapping pairs than halos (the scan is repeated with room for all) and more than a workgroup's
list holds (entries written one by one), against the oracle; a second call finds the room there."""
import numpy as np
import pytest

from test_gpu_merge import check

pytestmark = pytest.mark.gpu


def records(xyz, r, seed):
    rec = np.random.default_rng(seed).normal(size=(len(xyz), 11)).astype(np.float32)
    rec[:, :3] = xyz
    rec[:, 6] = r
    return rec


def nested(n):
    """Every halo near one centre: n (n - 1) / 2 containments or so."""
    rng = np.random.default_rng(n)
    return records(rng.normal(scale=0.5, size=(n, 3)), 3.0 + rng.uniform(size=n), n)


def lattice(m):
    """Halos 1.1 radii apart: some 13 overlapping pairs each, no containment."""
    i = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return records(1.1 * i + 0.001 * np.random.default_rng(m).uniform(size=i.shape), 1.0, m)


def shell(n):
    """A large halo with n small ones just outside its centre's reach, and all of them cut by it."""
    k = np.arange(n) + 0.5
    phi, z = np.pi * (1 + 5**0.5) * k, 1 - 2 * k / n
    s = np.sqrt(1 - z * z)
    xyz = 60.3 * np.stack([s * np.cos(phi), s * np.sin(phi), z], -1)
    return records(np.concatenate([[[0, 0, 0]], xyz]), np.concatenate([[60.0], np.full(n, 0.7)]), n)


@pytest.mark.parametrize("rec", [nested(17), nested(900), lattice(7), lattice(20), shell(3000)],
                         ids=["nested17", "nested900", "lattice7", "lattice20", "shell3000"])
@pytest.mark.parametrize("ties", [False, True])
def test_lists_run_over(oracle, rec, ties):
    from huntian_hip import api

    api.context(0).release_scratch()
    check(oracle, rec, True, ties)
    check(oracle, rec, True, ties)
