"""Compaction of the active particles of large systems, on both sides of the size
where a scan of the blocks' counts takes over: the right particles get their
forces, and the time grows with the size, not with its square (needs an
MI355X).

Tolerance: unsoftened FP32 pair terms carry a few eps = 6e-8 each, so a sum is
within 1e-6 of the sum of its terms' magnitudes.
"""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

I64 = C.POINTER(C.c_int64)
SCAN_FROM = (1 << 14) * 256   # particles


def _context(pkg, n, pos, mass, active):
    call = pkg._native.call
    ctx = pkg._native.Context(n, pkg._native.MODES["split"])
    ctx.set_params(1.0, [1e-9] * 6)
    ctx.upload(pos, None, mass)
    ctx.upload_acc(np.full((n, 3), 7.0))
    call("nb_adaptive_init", ctx.handle, 1e-6, 1 << 20, 0.025, 0.0, 1.0)
    te, tb = np.where(active, 64, 128).astype(np.int64), np.zeros(n, dtype=np.int64)
    call("nb_adaptive_set_steps", ctx.handle, te.ctypes.data_as(I64), tb.ctypes.data_as(I64))
    return ctx


@pytest.mark.parametrize("n", [SCAN_FROM - 256, SCAN_FROM - 255, SCAN_FROM + 1025 * 256 + 77])
def test_active_particles_of_a_large_system(pkg, n):
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3))
    mass = np.full(n, 1.0 / n)
    active = rng.random(n) < 5e-4
    active[[0, 255, 256, n - 1]] = True
    active[1000 * 256:1100 * 256] = False       # blocks without any
    active[5000 * 256:5001 * 256] = True        # and a full one
    with _context(pkg, n, pos, mass, active) as ctx:
        na = C.c_int64()
        pkg._native.call("nb_adaptive_compute_force", ctx.handle, 64, C.byref(na))
        acc = ctx.download(pos=False, vel=False)["acc"]
    assert na.value == active.sum()
    assert np.all(acc[~active] == 7.0) and not np.any(np.all(acc[active] == 7.0, axis=1))
    which = np.flatnonzero(active)
    for i in np.concatenate([which[:3], which[len(which) // 2:][:3], which[-3:]]):
        d = pos - pos[i]
        r2 = np.einsum("ij,ij->i", d, d)
        r2[i] = np.inf
        w = mass / (r2 * np.sqrt(r2))
        err = np.linalg.norm(acc[i] - w @ d)
        assert err <= 1e-6 * np.sum(w * np.sqrt(np.where(np.isfinite(r2), r2, 0.0))), i


def test_compaction_time_is_linear(pkg):
    times = []
    for n in (1 << 23, 1 << 25):
        pos = np.random.default_rng(1).random((n, 3))
        with _context(pkg, n, pos, np.full(n, 1.0 / n), np.zeros(n, dtype=bool)) as ctx:
            na = C.c_int64()
            t = []
            for _ in range(6):
                a = time.perf_counter()
                pkg._native.call("nb_adaptive_compute_force", ctx.handle, 65, C.byref(na))   # none active
                t.append(time.perf_counter() - a)
            assert na.value == 0
            times.append(min(t))
    assert times[1] < 6.0 * times[0], times     # four times the particles
