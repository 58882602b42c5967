"""The FP64 pair kernel against the FP64 oracle where its fast Newtonian terms,
its softening window and its split of the sources over waves can go wrong
(needs an MI355X).

Tolerance: a Newtonian term carries at most about 8 half-ulp roundings, a
spline term the roundings of polynomial terms that add up to 120 times its value
near u = 1 (400 half ulps), and the sum of n terms at most n more, so with both
sides' roundings |a - a_ref| <= 2 (n + 8) 2^-53 sum |terms| without softening
and 2 (n + 400) 2^-53 sum |terms| with it, per component.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(rng, n, kind):
    pos = rng.standard_normal((n, 3))
    mass = rng.uniform(0.5, 2.0, n) / n
    if kind == "close" and n > 3:      # coincident, at 1e-80 and at 1e-60 from one another
        pos[1] = pos[0]
        pos[2] = pos[0] = pos[1] = 0.0
        pos[2, 0], pos[3] = 1e-80, [0.0, 1e-60, 0.0]
    if kind == "far" and n > 2:        # r^2 overflows
        pos[-1] = [1e160, 0.0, -1e155]
    if kind == "heavy":
        mass *= 1e60
    return pos, mass


@pytest.mark.parametrize("kind,h", [("plain", 0.01), ("plain", 0.0), ("soft", 5.0), ("mixed", 0.7),
                                    ("close", 1e-3), ("far", 0.01), ("heavy", 0.01)])
@pytest.mark.parametrize("n", [1, 3, 4, 63, 65, 257, 600])
def test_fp64_pairs_match_oracle(pkg, orc, n, kind, h):
    if h == 0.0 and kind != "plain":
        pytest.skip("coincident pairs need h > 0")
    pos, mass = _system(np.random.default_rng(n), n, kind)
    with pkg._native.Context(n, pkg._native.MODES["fp64"]) as ctx:
        ctx.set_params(1.0, [h] * 6)
        ctx.upload(pos, None, mass)
        ctx.compute_force()
        acc = ctx.download(pos=False, vel=False)["acc"]
        ctx.compute_potential(self_term=False)
        pot = ctx.download(pos=False, vel=False, acc=False, pot=True)["pot"]
        probe = ctx.force_at_points(pos[: n // 2 + 1], h)
    size = np.zeros((n, 3))
    size_pot = np.zeros(n)
    for j in range(n):
        s = np.abs(orc.force_at_points(pos, h, pos[j:j + 1], mass[j:j + 1]))
        q = np.abs(orc.potential_at_points(pos, h, pos[j:j + 1], mass[j:j + 1]))
        same = np.all(pos == pos[j], axis=1)
        s[same], q[same] = 0.0, 0.0
        size += s
        size_pot += q
    ref = orc.compute_force(pos, mass, [h] * 6, 1.0, skip_self=h == 0.0)
    pref = orc.compute_potential(pos, mass, [h] * 6, 1.0, skip_self=h == 0.0)
    tol = 2 * (n + (400 if h > 0.0 else 8)) * 2.0 ** -53
    assert np.all(np.abs(acc - ref) <= tol * size)
    assert np.all(np.abs(pot - pref) <= tol * size_pot)
    if h > 0.0:   # (the oracle's probe on a particle is NaN without softening)
        assert np.all(np.abs(probe - ref[: n // 2 + 1]) <= tol * size[: n // 2 + 1])
