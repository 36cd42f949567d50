"""The offsets of the shell blocks (scan_counts in csrc/shell_analyse.hip): sums of 32-bit counts
beyond 2^31 and 2^32, one count, and a number of counts that is no multiple of anything."""
import ctypes as C

import numpy as np
import pytest

from huntian_hip import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count", [(1, 7), (1000, 3), (3_000_001, 755), (1_000_003, 5001)])
def test_offsets_in_64_bits(n, count):
    import torch

    ctx = api.context(0)
    scan = ctx.lib._ZN3hnt11scan_countsEP7hnt_ctxPKiPll
    scan.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64]
    rng = np.random.default_rng(n)
    cnt = rng.integers(count - 1, count + 2, n).astype(np.int32)
    dev = torch.as_tensor(cnt, device="cuda")
    off = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    assert scan(ctx.handle, dev.data_ptr(), off.data_ptr(), n) == 0
    want = np.concatenate([[0], np.cumsum(cnt.astype(np.int64))[:-1]])
    assert np.array_equal(off.cpu().numpy(), want)
