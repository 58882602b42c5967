"""Active subsets of a block step at the edges of waves and blocks: the ordered
compaction, the force of the active particles alone, and the kick with the
reduction of the timeline it leaves (needs an MI355X).

Tolerance: unsoftened FP32 pair terms carry a few eps = 6e-8 each, so a sum is
within 1e-6 of the sum of its terms' magnitudes (FP64 mode: 1e-12).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

I64 = C.POINTER(C.c_int64)


@pytest.mark.parametrize("mode,tol", [("split", 1e-6), ("fp32", 1e-6), ("fp64", 1e-12)])
@pytest.mark.parametrize("which", ["first", "last", "some", "all_but_one"])
@pytest.mark.parametrize("n", [2, 64, 65, 256, 257, 1025])
def test_active_subset_and_kick(pkg, orc, mode, tol, which, n):
    call = pkg._native.call
    rng = np.random.default_rng(n)
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    if mode == "fp32":
        pos, vel, mass = (v.astype(np.float32).astype(np.float64) for v in (pos, vel, mass))
    active = rng.random(n) < 0.3
    if which in ("first", "last"):
        active[:] = False
    if which == "all_but_one":
        active[:] = True
    active[0 if which == "first" else n - 1] = which != "all_but_one"
    h, interval, base, t = 1e-7, 1e-6, 1 << 20, 64
    te, tb = np.where(active, t, 2 * t).astype(np.int64), np.zeros(n, dtype=np.int64)
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, vel, mass)
        ctx.compute_force()
        call("nb_adaptive_init", ctx.handle, interval, base, 0.025, 0.0, 1.0)
        call("nb_adaptive_set_steps", ctx.handle, te.ctypes.data_as(I64), tb.ctypes.data_as(I64))
        ctx.upload_acc(np.full((n, 3), 7.0))
        na, first, nxt = C.c_int64(), C.c_int64(), C.c_int64()
        call("nb_adaptive_compute_force", ctx.handle, t, C.byref(na))       # count read back
        a1 = ctx.download(pos=False, vel=False)["acc"]
        call("nb_adaptive_min_endstep", ctx.handle, C.byref(first))
        call("nb_adaptive_compute_force", ctx.handle, t, C.byref(na))       # count known
        d = ctx.download(pos=False, vel=True)
        call("nb_adaptive_kick", ctx.handle, t)
        call("nb_adaptive_min_endstep", ctx.handle, C.byref(nxt))
        te2, tb2 = np.zeros(n, dtype=np.int64), np.zeros(n, dtype=np.int64)
        call("nb_adaptive_get_steps", ctx.handle, te2.ctypes.data_as(I64), tb2.ctypes.data_as(I64))
        v2 = ctx.download(pos=False, vel=True, acc=False)["vel"]
    acc = d["acc"]
    ref = orc.compute_force(pos, mass, [h] * 6)
    mag = np.zeros(n)
    for j in range(n):
        s = np.linalg.norm(orc.force_at_points(pos, h, pos[j:j + 1], mass[j:j + 1]), axis=1)
        s[j] = 0.0
        mag += s
    assert na.value == active.sum() and first.value == t
    assert np.array_equal(a1, acc) and np.all(acc[~active] == 7.0)
    assert np.all(np.linalg.norm(acc - ref, axis=1)[active] <= tol * mag[active])
    step = orc.get_timestep(acc, np.full(n, h), err_tol=0.025, min_step=0.0, max_step=1.0,
                            time_interval=interval, time_base=base)
    assert np.array_equal(te2, np.where(active, t + step, 2 * t))
    assert np.array_equal(tb2, np.where(active, t, 0)) and nxt.value == te2.min()
    dt = np.where(active, (t + 0.5 * step - 0.5 * t) * interval, 0.0)
    eps = 2.0 ** -22 if mode == "fp32" else 2.0 ** -51     # an FP32 / FP64 product and sum
    want = d["vel"] + acc * dt[:, None]
    assert np.all(np.abs(v2 - want) <= eps * (np.abs(d["vel"]) + np.abs(acc * dt[:, None])))
