"""hnt_merge_catalog with memory for its results but not for the first guess at the number of
containments and overlapping pairs (80 bytes a halo): they are counted first, and the catalog is the
same as with all memory free."""
import numpy as np
import pytest
import torch

from huntian_hip import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [20000.0, 900.0])
def test_little_memory(side):
    n = 4_000_000
    rng = np.random.default_rng(7)
    rec = np.zeros((n, 11), np.float32)
    rec[:, :3] = rng.uniform(0, side, (n, 3))
    rec[:, 6] = 1.0 + 0.5 * rng.uniform(size=n)
    rec = torch.as_tensor(rec, device="cuda")
    ctx = api.context(0)
    want = api.merge_catalog(rec, volume_reduction=True).cpu()
    ctx.release_scratch()
    torch.cuda.empty_cache()
    # the call's output takes 176 MB, its scratch 690 with the guess and 370 to 440 without
    left = 700_000_000
    hog = []
    try:
        for _ in range(3):  # the driver's figure moves with the first of them
            more = torch.cuda.mem_get_info()[0] - left
            if more > 50_000_000:
                hog.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
        print(f"side {side}: {torch.cuda.mem_get_info()[0] / 1e6:.0f} MB free", flush=True)
        assert torch.cuda.mem_get_info()[0] < 1.1 * left
        got = api.merge_catalog(rec, volume_reduction=True)
        print(f"{torch.cuda.mem_get_info()[0] / 1e6:.0f} MB left", flush=True)
    finally:
        hog.clear()
        torch.cuda.empty_cache()
        ctx.release_scratch()
    assert torch.equal(got.cpu(), want) and len(want) < n
