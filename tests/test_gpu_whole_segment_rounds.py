"""Launches whose waves walk whole segments (32768 targets and more) take enough
segments that their last round of workgroups is a small part of them: the
allocation-free call and large active subsets are as fast as a context's force
on the same particles in 64 segments (needs an MI355X)."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

I64 = C.POINTER(C.c_int64)


def _best(f, sync, k=12):
    f()
    sync()
    t = []
    for _ in range(k):
        a = time.perf_counter()
        f()
        sync()
        t.append(time.perf_counter() - a)
    return min(t)


def test_allocation_free_call(pkg):
    import torch
    nat = pkg._native
    n = 200000
    pos, vel, mass = pkg.ics.plummer(n, seed=3)
    with nat.Context(n, nat.MODES["split"]) as ctx:
        ctx.set_params(1.0, [0.01] * 6)
        ctx.upload(pos, vel, mass)
        ctx.set_tuning(1, 64, 0, 0)     # no sort: the order given, as in the call below
        force = _best(ctx.compute_force, ctx.sync)
    t = [torch.tensor(np.ascontiguousarray(pos[:, k]), device="cuda") for k in range(3)]
    t.append(torch.tensor(mass, device="cuda"))
    o = [torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(3)]
    call = _best(lambda: nat.compute_force_noalloc(nat.NB_MODE_SPLIT, n, *[v.data_ptr() for v in t + o],
                                                   h_const=0.01), torch.cuda.synchronize)
    assert call < 1.08 * force, (call, force)     # 1.2 in the three segments of old


def test_large_active_subset(pkg):
    nat = pkg._native
    n = 50000
    pos, vel, mass = pkg.ics.plummer(n, seed=3)
    with nat.Context(n, nat.MODES["split"]) as ctx:
        ctx.set_params(1.0, [0.01] * 6)
        ctx.upload(pos, vel, mass)
        ctx.set_tuning(1, 64, 16, 0)
        ctx.compute_force()
        ctx.set_tuning(1, 64, 0, 0)
        force = _best(ctx.compute_force, ctx.sync)
        nat.call("nb_adaptive_init", ctx.handle, 1e-6, 1 << 20, 0.025, 0.0, 1.0)
        te = np.where(np.arange(n) % 100 != 7, 64, 128).astype(np.int64)
        tb = np.zeros(n, dtype=np.int64)
        nat.call("nb_adaptive_set_steps", ctx.handle, te.ctypes.data_as(I64), tb.ctypes.data_as(I64))
        na = C.c_int64()
        subset = _best(lambda: nat.call("nb_adaptive_compute_force", ctx.handle, 64, C.byref(na)), ctx.sync)
    assert na.value == 99 * n // 100
    assert subset < 1.08 * force, (subset, force)
