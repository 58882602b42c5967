"""Downloads into pinned host memory of the caller's: whole arrays, alone and
beside pageable ones, large ones by a copy command that needs no host thread to
move the bytes (needs an MI355X).
"""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

PIECE = 1 << 17   # doubles


def _pinned(n):
    # (filled by numpy: torch would leave its OpenMP threads spinning into the timing)
    a = torch.empty((n, 3), dtype=torch.float64, pin_memory=True).numpy()
    a[:] = -1.0
    return a


@pytest.mark.parametrize("n", [1, PIECE // 3, PIECE // 3 + 1, 400003])
def test_pinned_and_pageable_arrays(pkg, n):
    nat = pkg._native
    rng = np.random.default_rng(n)
    want = [rng.standard_normal((n, 3)) for _ in range(3)]
    with nat.Context(n, nat.MODES["fp64"]) as ctx:
        ctx.upload(want[0], want[1], np.ones(n))
        ctx.upload_acc(want[2])
        for kinds in ("ppp", "pmp", "mpm", "mmm"):
            got = [_pinned(n) if k == "p" else np.full((n, 3), -1.0) for k in kinds]
            nat.call("nb_download", ctx.handle, *[nat.dptr(g) for g in got], None)
            for a, b in zip(got, want):
                assert np.array_equal(a, b), kinds


def test_large_pinned_arrays_take_one_thread(pkg):
    nat = pkg._native
    n = 1 << 21
    pos = np.random.default_rng(1).standard_normal((n, 3))
    with nat.Context(n, nat.MODES["fp64"]) as ctx:
        ctx.upload(pos, pos, np.ones(n))
        a, b = _pinned(n), _pinned(n)
        nat.call("nb_download", ctx.handle, nat.dptr(a), nat.dptr(b), None, None)
        wall, cpu = time.perf_counter(), time.process_time()
        for _ in range(40):     # about 0.1 s
            nat.call("nb_download", ctx.handle, nat.dptr(a), nat.dptr(b), None, None)
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert np.array_equal(a, pos) and np.array_equal(b, pos)
    assert cpu < 2.0 * wall, (cpu, wall)
