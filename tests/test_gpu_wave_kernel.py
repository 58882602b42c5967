"""The wavefront force kernel (far path 0, one target per lane) at the edges of
waves, quarters and segments, against the FP64 oracle (needs an MI355X).

Tolerance: an unsoftened FP32 pair term carries a few eps = 6e-8, so a sum is
within 1e-6 of the sum of its terms' magnitudes.  A softened term near u = 1 is
the sum of polynomial terms 120 times its value, so with softened pairs it is
1e-6 plus 3e-5 of the softened terms' magnitudes (120 x 4 eps).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL, TOL_SOFT = 1e-6, 3e-5


def _bounds(orc, pos, mass, h):
    n = len(mass)
    size, size_pot = np.zeros(n), np.zeros(n)
    for j in range(n):
        s = np.linalg.norm(orc.force_at_points(pos, h, pos[j:j + 1], mass[j:j + 1]), axis=1)
        q = np.abs(orc.potential_at_points(pos, h, pos[j:j + 1], mass[j:j + 1]))
        r = np.linalg.norm(pos - pos[j], axis=1)
        s[r == 0], q[r == 0] = 0.0, 0.0
        w = np.where(r <= h * (1 + 1e-6), TOL_SOFT, TOL)
        size += w * s
        size_pot += w * q
    return size, size_pot


@pytest.mark.parametrize("mode", ["split", "fp32"])
@pytest.mark.parametrize("h", [1e-3, 0.3])
@pytest.mark.parametrize("n,nseg", [(2, 1), (63, 1), (65, 3), (129, 1), (255, 2), (1000, 5), (1025, 16)])
def test_wave_kernel_forces_and_potentials(pkg, orc, mode, h, n, nseg):
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    mass = mass * np.random.default_rng(n).uniform(0.0, 2.0, n)
    mass[n // 2] = 0.0
    pos = pos + [3.0, -2.0, 1.0]
    if mode == "fp32":
        pos, mass = (v.astype(np.float32).astype(np.float64) for v in (pos, mass))
    size, size_pot = _bounds(orc, pos, mass, h)
    ref, pref = orc.compute_force(pos, mass, [h] * 6), orc.compute_potential(pos, mass, [h] * 6)
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, vel, mass)
        ctx.set_tuning(1, nseg, 16, 0)
        ctx.compute_force()
        ctx.compute_potential(self_term=False)
        d = ctx.download(pos=False, vel=False, acc=True, pot=True)
    assert np.all(np.linalg.norm(d["acc"] - ref, axis=1) <= size)
    assert np.all(np.abs(d["pot"] - pref) <= size_pot)


@pytest.mark.parametrize("n", [64, 1000])
def test_wave_kernel_skips_central_sources(pkg, orc, n):
    """Central bodies are left to the FP64 pass wherever the sort puts them."""
    pos, vel, mass = pkg.ics.plummer(n, seed=3)
    mass[:2] = [5.0, 3.0]
    h = 1e-3
    size, _ = _bounds(orc, pos, mass, h)
    ref = orc.compute_force(pos, mass, [h] * 6)
    with pkg._native.Context(n, pkg._native.MODES["split_central"]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, vel, mass)
        ctx.set_central(2)
        ctx.set_tuning(1, 4, 16, 0)
        ctx.compute_force()
        acc = ctx.download(pos=False, vel=False)["acc"]
    assert np.all(np.linalg.norm(acc - ref, axis=1) <= size)
