"""The neighbour scans of hnt_merge_catalog where most entries are past a workgroup's list: lanes of
a wavefront then take their places in the output together.  Against the oracle."""
import numpy as np
import pytest

from test_gpu_merge import check
from test_gpu_merge_scan import nested, records

pytestmark = pytest.mark.gpu


def shells(n, m):
    """m large halos beside one another, each with n small ones around it, all overlapping."""
    rng = np.random.default_rng(n)
    d = rng.normal(size=(m, n, 3))
    d *= 6.2 / np.linalg.norm(d, axis=2, keepdims=True)
    c = np.arange(m)[:, None] * np.array([[9.0, 0.0, 0.0]])
    xyz = np.concatenate([c, (c[:, None] + d).reshape(-1, 3)])
    return records(xyz, np.concatenate([np.full(m, 6.0), np.full(n * m, 0.5)]), n)


@pytest.mark.parametrize("rec", [nested(2500), shells(400, 12), shells(33, 1)],
                         ids=["nested2500", "shells400", "shells33"])
def test_entries_past_the_list(oracle, rec):
    from huntian_hip import api

    api.context(0).release_scratch()
    check(oracle, rec, True, False)
    check(oracle, rec, True, False)
