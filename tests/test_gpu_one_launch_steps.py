"""Captured KDK steps that run in one launch each (far path 0, fewer than 32768
particles) give the bits of the same steps launched one kernel at a time, where
64-target groups, tiles and segments end raggedly (needs an MI355X).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(pkg, mode, n, steps, dt, use_graph, central=0, runs=1):
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    if central:
        mass[:central] = 0.1
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [0.05] * 6)
        ctx.upload(pos, vel, mass)
        if central:
            ctx.set_central(central)
        ctx.compute_force()
        ctx.half_kick(+1, dt)
        for k in range(runs):
            ctx.kdk_steps(steps, dt, k * steps * dt, use_graph=use_graph)
        return ctx.download(pos=True, vel=True, acc=True)


@pytest.mark.parametrize("mode,central", [("split", 0), ("fp32", 0), ("split_central", 0), ("split_central", 3)])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 257, 1000, 4097, 32767])
def test_one_launch_steps_match_single_launches(pkg, mode, central, n):
    if central >= n:
        pytest.skip("needs more particles than central bodies")
    steps, dt, runs = 4, 1e-3, 2
    a = _run(pkg, mode, n, steps, dt, True, central, runs)
    b = _run(pkg, mode, n, steps, dt, False, central, runs)
    assert all(np.array_equal(a[k], b[k]) for k in a)


@pytest.mark.parametrize("mode", ["split", "fp32"])
def test_one_launch_steps_repeat(pkg, mode):
    """The workgroup that arrives last differs from run to run, the sums do not."""
    a = _run(pkg, mode, 5000, 16, 1e-3, True, runs=3)
    for _ in range(2):
        b = _run(pkg, mode, 5000, 16, 1e-3, True, runs=3)
        assert all(np.array_equal(a[k], b[k]) for k in a)
