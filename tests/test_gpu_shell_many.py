"""The shell analysis of very many peaks (from 2^18 on the crossing pass and the walk take four lanes per
peak and the far gather a field per launch) against the lane-per-peak kernel, bit for bit: shells
beyond a brick's halo, peaks whose balls leave the grid, and counts on both sides of the line."""
import pytest

from test_gpu_shell_blocks import _compare, _fields, _peaks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nhunt,count,variant,lapd,lo", [
    (160, 13, (1 << 18) + 77, "C", False, 14), (160, 13, (1 << 18) - 1, "C", False, 14),
    (96, 12, 270_000, "A", True, 2), (97, 9, 263_001, "B", False, 0)])
def test_many_peaks(websky, n, nhunt, count, variant, lapd, lo):
    _compare(_fields(n, 3 + n, lapd), _peaks(n, count, 5 + n, lo, n - lo), n, nhunt, websky, variant,
             f"{n} {count} {variant}")
