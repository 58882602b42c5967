"""KDK steps with more central bodies than the step's kick adds up itself: values
around that count, captured and eager alike, and the time, which follows the
force's FP64 pass and not one lane per target (needs an MI355X).

Tolerance: an FP32 pair term is within 1e-6 of its size where unsoftened (h is
below every separation here), so a step changes a velocity by at most
1e-6 dt sum |terms| too much, with the terms' sum taken at twice its initial
value for the motion of the run, and positions by that times the run's time.
"""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(pkg, n, ncentral, nsteps, dt, use_graph, pos, vel, mass):
    with pkg._native.Context(n, pkg._native.MODES["split_central"]) as ctx:
        ctx.set_params(1.0, [1e-7] * 6)
        ctx.upload(pos, vel, mass)
        ctx.set_central(ncentral)
        ctx.set_tuning(1, 8, 16, 0)
        ctx.kdk_steps(nsteps, dt, 0.3, use_graph=use_graph)
        return ctx.download(pos=True, vel=True, acc=True)


@pytest.mark.parametrize("n,ncentral", [(257, 16), (257, 17), (1000, 100), (300, 300)])
def test_steps_with_many_central_bodies(pkg, orc, n, ncentral):
    dt, nsteps, tol = 1e-4, 16, 1e-6
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    a = _run(pkg, n, ncentral, nsteps, dt, True, pos, vel, mass)
    b = _run(pkg, n, ncentral, nsteps, dt, False, pos, vel, mass)
    assert all(np.array_equal(a[k], b[k]) for k in a)
    p, v, _ = orc.kdk_steps(pos, vel, mass, [1e-7] * 6, 1.0, nsteps=nsteps, dt=dt, t_begin=0.3)
    mag = np.zeros(n)
    for j in range(n):
        s = np.linalg.norm(orc.force_at_points(pos, 1e-7, pos[j:j + 1], mass[j:j + 1]), axis=1)
        s[j] = 0.0
        mag += s
    dv = 2 * tol * nsteps * dt * mag + nsteps * 2.0 ** -51 * np.linalg.norm(v, axis=1)
    dx = nsteps * dt * dv + nsteps * 2.0 ** -51 * np.linalg.norm(p, axis=1)
    assert np.all(np.linalg.norm(a["vel"] - v, axis=1) <= dv)
    assert np.all(np.linalg.norm(a["pos"] - p, axis=1) <= dx)


def test_step_time_follows_the_force(pkg):
    n, ncentral, nsteps = 4097, 1024, 16
    pos, vel, mass = pkg.ics.plummer(n, seed=1)
    with pkg._native.Context(n, pkg._native.MODES["split_central"]) as ctx:
        ctx.set_params(1.0, [0.01] * 6)
        ctx.upload(pos, vel, mass)
        ctx.set_central(ncentral)
        ctx.set_tuning(1, 64, 0, 0)

        def best(f):
            f()
            t = []
            for _ in range(5):
                a = time.perf_counter()
                f()
                ctx.sync()
                t.append(time.perf_counter() - a)
            return min(t)

        force = best(lambda: [ctx.compute_force() for _ in range(nsteps)])
        steps = best(lambda: ctx.kdk_steps(nsteps, 1e-6, 0.0, use_graph=True))
    # a step is a force, a kick and a drift; one lane per target took four times as long
    assert steps < 2.0 * force, (steps, force)
