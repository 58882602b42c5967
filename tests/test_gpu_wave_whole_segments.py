"""The wavefront kernel from 32768 targets on, where every wave has 64 targets of
its own and walks whole segments, on a context's own particles (needs an
MI355X): forces and potentials of sampled particles against FP64 sums.

Tolerance: an unsoftened FP32 pair term carries a few eps = 6e-8, so a sum is
within 1e-6 of the sum of its terms' magnitudes.  A softened term is the sum of
polynomial terms 120 times its value near u = 1: 3e-5 of its magnitude, which
is below that of the Newtonian term at the larger of r and h / 2.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL, TOL_SOFT = 1e-6, 3e-5


def _sample(orc, pos, mass, h, which):
    ref = orc.force_at_points(pos[which], h, pos, mass)
    pref = orc.potential_at_points(pos[which], h, pos, mass)
    size, size_pot = np.zeros(len(which)), np.zeros(len(which))
    for k, i in enumerate(which):
        r = np.linalg.norm(pos - pos[i], axis=1)
        w = np.where(r <= h * (1 + 1e-6), TOL_SOFT, TOL) * mass
        w[i] = 0.0
        r = np.maximum(r, 0.5 * h)
        size[k], size_pot[k] = np.sum(w / r ** 2), np.sum(w / r)
    # (the oracle's potential at a particle's own place has its self term)
    pref -= orc.potential_at_points(pos[which[:1]], h, pos[which[:1]], np.ones(1)) * mass[which]
    return ref, pref, size, size_pot


@pytest.mark.parametrize("mode", ["split", "fp32", "split_central"])
@pytest.mark.parametrize("n,nseg,h", [(32768, 1, 1e-3), (32769, 7, 0.05), (40001, 64, 1e-3)])
def test_own_particles_with_whole_segments(pkg, orc, mode, n, nseg, h):
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    pos = pos + [3.0, -2.0, 1.0]
    if mode == "fp32":
        pos, mass = (v.astype(np.float32).astype(np.float64) for v in (pos, mass))
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, vel, mass)
        if mode == "split_central":
            ctx.set_central(2)
        ctx.set_tuning(1, nseg, 16, 0)
        ctx.compute_force()
        ctx.compute_potential(self_term=False)
        d = ctx.download(pos=False, vel=False, acc=True, pot=True)
    which = np.concatenate([[0, 1, n - 2, n - 1], np.random.default_rng(n).integers(0, n, 300)])
    ref, pref, size, size_pot = _sample(orc, pos, mass, h, which)
    assert np.all(np.linalg.norm(d["acc"][which] - ref, axis=1) <= size)
    assert np.all(np.abs(d["pot"][which] - pref) <= size_pot)
