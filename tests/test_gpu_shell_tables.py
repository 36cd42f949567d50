"""Shell tables that list a shell's cells in another order than build_shell_tables does: a shell is
summed in the order given, by shell blocks (no cell records: 32 bytes per cell less memory) as by the
lane-per-peak kernel (plain order), bit for bit."""
import dataclasses

import numpy as np
import pytest
import torch

from huntian_hip import api
from test_gpu_shell_blocks import _fields, _peaks, _same

pytestmark = pytest.mark.gpu


def _reordered(tab, order):
    q = np.concatenate([s + order(c) for s, c in zip(tab.shell_start, tab.shell_count)])
    return dataclasses.replace(tab, **{k: np.ascontiguousarray(getattr(tab, k)[q])
                                       for k in ("di", "dj", "dk")})


@pytest.mark.parametrize("name,order", [
    ("as built", np.arange), ("reversed", lambda c: np.arange(c)[::-1]),
    ("shuffled", lambda c: np.random.default_rng(c).permutation(c))])
def test_any_order_within_a_shell(websky, name, order):
    n, nhunt = 128, 12
    f, pk = _fields(n, 11, True), _peaks(n, 300, 12)
    tab = _reordered(api.build_shell_tables(nhunt), order)

    def run(how):
        return api.shell_analyse(f, pk["pi"], pk["pj"], pk["pk"], pk["Rf"], pk["ir2min"], tab, websky,
                                 alatt=2.0, ZZon=1.0, fcrit=api.fsc_of_z(websky, 0.0), order=how)

    plain = run("plain")
    ctx = api.context(0)
    run("crossing")
    ctx.release_scratch()
    free = torch.cuda.mem_get_info()[0]
    got = run("crossing")
    used = free - torch.cuda.mem_get_info()[0]
    ctx.release_scratch()
    print(name, used, flush=True)
    _same(got, plain, name)
    assert used < 32 * n ** 3
