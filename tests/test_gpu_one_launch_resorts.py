"""One-launch KDK steps across re-sorts (needs an MI355X): 16-step graphs with a
re-sort before each and an eager remainder.  A uniform field of strength zero
sends the same steps through force, sums, field and kick one launch at a time,
with the re-sorts at the same places; the results have the same bits (with
central bodies the two take their FP64 terms from different kernels: a few
roundings of 2^-53 a step, held to 1e-11 of the largest value).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(pkg, mode, n, central, nsteps, field):
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    if central:
        mass[:central] = 0.1
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [0.05] * 6)
        ctx.upload(pos, vel, mass)
        if central:
            ctx.set_central(central)
        if field:
            ctx.add_background(4, [0.0, 0.0, 0.0])
        ctx.set_tuning(1, 16, 16, 0)
        ctx.compute_force()
        ctx.half_kick(+1, 2e-3)
        for k in range(2):
            ctx.kdk_steps(nsteps, 2e-3, k * nsteps * 2e-3, use_graph=True)
        return ctx.download(pos=True, vel=True, acc=True)


@pytest.mark.parametrize("mode,central", [("split", 0), ("fp32", 0), ("split_central", 0), ("split_central", 3)])
@pytest.mark.parametrize("n,nsteps", [(65, 35), (1000, 48), (4097, 35), (9001, 35)])
def test_steps_across_resorts(pkg, mode, central, n, nsteps):
    a = _run(pkg, mode, n, central, nsteps, False)
    b = _run(pkg, mode, n, central, nsteps, True)
    for k in a:
        if central:
            assert np.max(np.abs(a[k] - b[k])) <= 1e-11 * np.max(np.abs(b[k])), k
        else:
            assert np.array_equal(a[k], b[k]), k
