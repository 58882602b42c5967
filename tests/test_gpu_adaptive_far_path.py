"""Active subsets of 2^14 particles and more take the context's far path 4 (stored
target geometry, source weights, and with an FP64 state the far and near
passes), with the sums written straight to the particles or, where something
follows, gathered first (needs an MI355X).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

I64 = C.POINTER(C.c_int64)


def _run(pkg, mode, far, extra, pos, vel, mass, active):
    call = pkg._native.call
    n = len(mass)
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [0.002] * 6)
        ctx.upload(pos, vel, mass)
        if extra == "central":
            ctx.set_central(2)
        if extra == "field":
            ctx.add_background(4, [0.25, 0.0, -0.5])
        ctx.set_tuning(1, 4, 0, far)
        ctx.compute_force()
        call("nb_adaptive_init", ctx.handle, 1e-3, 1 << 10, 1e-2, 0.0, 1.0)
        te, tb = np.where(active, 64, 128).astype(np.int64), np.zeros(n, dtype=np.int64)
        call("nb_adaptive_set_steps", ctx.handle, te.ctypes.data_as(I64), tb.ctypes.data_as(I64))
        out = []
        for _ in range(2):
            ctx.upload_acc(np.full((n, 3), 7.0))
            na = C.c_int64()
            call("nb_adaptive_compute_force", ctx.handle, 64, C.byref(na))
            assert na.value == active.sum()
            out.append(ctx.download(pos=False, vel=False)["acc"])
    assert np.array_equal(out[0], out[1])
    return out[0]


@pytest.mark.parametrize("mode,extra", [("split", None), ("fp32", None), ("split", "field"),
                                        ("split_central", "central")])
@pytest.mark.parametrize("nactive", [1 << 14, 20003])
def test_large_active_subset_far_path_4(pkg, orc, mode, extra, nactive):
    pos, vel, mass = pkg.ics.collision(16001, seeds=(7, 8))
    n = len(mass)
    active = np.zeros(n, dtype=bool)
    active[np.random.default_rng(1).choice(n, nactive, replace=False)] = True
    if mode == "fp32":
        pos, mass = (v.astype(np.float32).astype(np.float64) for v in (pos, mass))
    ref = orc.compute_force(pos, mass, [0.002] * 6)
    if extra == "field":
        ref = ref + [0.25, 0.0, -0.5]
    acc = _run(pkg, mode, 4, extra, pos, vel, mass, active)
    valu = _run(pkg, mode, 0, extra, pos, vel, mass, active)
    assert np.all(acc[~active] == 7.0) and np.all(valu[~active] == 7.0)
    assert not np.array_equal(acc, valu)     # the matrix-core tiles, not far path 0
    # the bounds that far path 4 has on all particles of such a collision
    e = orc.rel_err(acc[active], ref[active])
    assert np.median(e) <= 2e-7 and np.percentile(e, 99) <= 2e-6
