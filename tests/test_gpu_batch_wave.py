"""The ensemble's wavefront kernel (far path 0, one target per lane) where its
systems end inside a wave, a quarter or a wave's part of the sources, with
eight waves per workgroup (few items) and with four, against the FP64 oracle
(needs an MI355X).

Tolerance: an unsoftened FP32 pair term carries a few eps = 6e-8, so a sum is
within 1e-6 of the sum of its terms' magnitudes.  A softened term near u = 1 is
the sum of polynomial terms 120 times its value: 3e-5 of its magnitude.
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


@pytest.mark.parametrize("mode", ["split", "split_central"])
@pytest.mark.parametrize("sizes,pad", [
    ([1, 2, 63, 64, 65, 255, 256, 257, 513, 1025], 0),
    ([511, 64, 1, 300], 1024),    # with 1024 pairs of particles beside: four waves per workgroup
])
def test_batch_wave_forces_and_potentials(pkg, orc, mode, sizes, pad):
    ns = np.array(sizes + [2] * pad, dtype=np.int64)
    off = np.concatenate([[0], np.cumsum(ns)])
    rng = np.random.default_rng(len(ns))
    pos, vel, _ = pkg.ics.plummer(int(off[-1]), seed=9)
    pos = pos + np.repeat(rng.uniform(-3.0, 3.0, (len(ns), 3)), ns, axis=0)
    mass = rng.uniform(0.0, 2.0, off[-1]) / np.repeat(ns, ns)
    mass[off[3]] = 0.0
    h = rng.choice([1e-3, 0.2], len(ns))
    G = rng.uniform(0.5, 2.0, len(ns))
    with pkg.Ensemble(off, mode) as e:
        e.set_params(G, h, 1e-3)
        e.upload(pos, vel, mass)
        if mode == "split_central":
            e.set_central(1)
        e.set_tuning(targets_per_thread=1, resident=0, far_path=0)
        e.compute_force()
        e.compute_potential()
        d = e.download(pos=False, vel=False, acc=True, pot=True)
    check = list(range(len(sizes))) + ([len(sizes), len(ns) - 1] if pad else [])
    for s in check:
        sl = slice(off[s], off[s + 1])
        size, size_pot = _bounds(orc, pos[sl], mass[sl], h[s])
        ref = orc.compute_force(pos[sl], mass[sl], [h[s]] * 6, G[s])
        pref = orc.compute_potential(pos[sl], mass[sl], [h[s]] * 6, G[s])
        assert np.all(np.linalg.norm(d["acc"][sl] - ref, axis=1) <= G[s] * size), s
        assert np.all(np.abs(d["pot"][sl] - pref) <= G[s] * size_pot), s
