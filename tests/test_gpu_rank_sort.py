"""The re-sort of a small system by ranks (up to 8192 particles), and of a larger
one by keys: every particle keeps its own data, also among particles with equal
keys, over several re-sorts (needs an MI355X).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["split", "fp32", "split_central"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 1000, 8191, 8192, 8193])
@pytest.mark.parametrize("places", [0, 5])   # particles on so few places (0: all apart)
def test_resort_keeps_every_particle(pkg, orc, mode, n, places):
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3))
    if places:
        pos = pos[rng.integers(0, min(places, n), n)]
    vel, mass = rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n) / n
    coll = rng.integers(1, 7, n).astype(np.uint8)
    pos, vel, mass = (v.astype(np.float32).astype(np.float64) for v in (pos, vel, mass))
    soft = [0.1, 0.2, 0.3, 0.4, 0.5, 0.6]
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, soft)
        ctx.upload(pos, vel, mass, coll)
        if mode == "split_central":
            ctx.set_central(2)
        ctx.set_tuning(1, 4, 1, 0)     # a re-sort before every force
        for _ in range(3):
            ctx.compute_force()
        d = ctx.download(pos=True, vel=True, acc=True)
    assert np.array_equal(d["pos"], pos) and np.array_equal(d["vel"], vel)
    # masses and softening lengths moved along: a mistaken one changes a force by
    # far more than 1e-4 of the largest, FP32 pair terms by a few 1e-6
    ref = orc.compute_force(pos, mass, soft, collection=coll)
    assert np.max(np.abs(d["acc"] - ref)) <= 1e-4 * np.max(np.abs(ref))
