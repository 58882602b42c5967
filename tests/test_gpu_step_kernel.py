"""KDK runs through the fused step kernel (kick with the segment sums and the
central bodies' FP64 terms, then the next drift) at the edges of its workgroups,
for odd and even step counts, eager and as graphs, against the FP64 oracle
(needs an MI355X).

Tolerance: an FP32 pair term is within 1e-6 of its size where unsoftened (h is
below every separation here), so a step changes a velocity by at most
1e-6 dt sum |terms| too much, with the terms' sum taken at twice its initial
value for the motion of the run, and positions by that times the run's time.
FP64 mode: 1e-12 in place of 1e-6.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,ncentral,tol", [("split", 0, 1e-6), ("split_central", 1, 1e-6),
                                               ("split_central", 3, 1e-6), ("fp64", 0, 1e-12)])
@pytest.mark.parametrize("nsteps,use_graph", [(1, False), (5, False), (2, True), (35, True)])
@pytest.mark.parametrize("n", [130, 256, 257, 1025])
def test_step_kernel_runs(pkg, orc, mode, ncentral, tol, nsteps, use_graph, n):
    h, dt, t0 = 1e-7, 1e-4, 0.3
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    mass[:ncentral] = 0.2
    acc0 = orc.compute_force(pos, mass, [h] * 6)
    v0 = orc.half_kick(vel, acc0, +1, dt)
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, v0, mass)
        if ncentral:
            ctx.set_central(ncentral)
        ctx.set_tuning(1, 8, 0 if mode == "fp64" else 3, 0)   # a re-sort within the run
        ctx.kdk_steps(nsteps, dt, t0, use_graph=use_graph)
        d = ctx.download(pos=True, vel=True, acc=True)
    p, v, a = orc.kdk_steps(pos, v0, mass, [h] * 6, 1.0, nsteps=nsteps, dt=dt, t_begin=t0)
    mag = np.zeros(n)
    for j in range(n):
        s = np.linalg.norm(orc.force_at_points(pos, h, pos[j:j + 1], mass[j:j + 1]), axis=1)
        s[j] = 0.0
        mag += s
    # (and the roundings of the state itself, one per step)
    dv = 2 * tol * nsteps * dt * mag + nsteps * 2.0 ** -51 * np.linalg.norm(v, axis=1)
    dx = nsteps * dt * dv + nsteps * 2.0 ** -51 * np.linalg.norm(p, axis=1)
    assert np.all(np.linalg.norm(d["vel"] - v, axis=1) <= dv)
    assert np.all(np.linalg.norm(d["pos"] - p, axis=1) <= dx)
