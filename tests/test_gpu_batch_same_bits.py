"""A system's forces and potentials have the same bits whatever other systems
share its ensemble (far path 0, one target per lane), on both sides of the
launch size where the workgroups go from eight waves to four (needs an MI355X).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 64, 257, 700, 1500, 2304, 5000]


@pytest.mark.parametrize("mode", ["split", "split_central"])
def test_bits_do_not_depend_on_the_other_systems(pkg, mode):
    rng = np.random.default_rng(4)
    ns = np.array(SIZES + [2] * 1024, dtype=np.int64)   # the pairs alone are 4096 workgroups
    off = np.concatenate([[0], np.cumsum(ns)])
    pos, vel, _ = pkg.ics.plummer(int(off[-1]), seed=3)
    # masses fall by 14 decades outwards, so that the tiles' sums do too: FP64 sums of
    # FP32 tile sums of one size are exact in any order, these are not
    mass = np.empty(off[-1])
    for a, b in zip(off[:-1], off[1:]):
        r = np.linalg.norm(pos[a:b], axis=1)
        mass[a:b] = 10.0 ** (-14.0 * np.argsort(np.argsort(r)) / (b - a))
    h = rng.choice([1e-3, 0.1], len(ns))

    def run(systems):
        o = off[:systems + 1]
        with pkg.Ensemble(o, mode) as e:
            e.set_params(1.0, h[:systems], 1e-3)
            e.upload(pos[:o[-1]], vel[:o[-1]], mass[:o[-1]])
            if mode == "split_central":
                e.set_central(1)
            e.set_tuning(targets_per_thread=1, resident=0, far_path=0)
            e.compute_force()
            e.compute_potential()
            return e.download(pos=False, vel=False, acc=True, pot=True)

    few, many = run(len(SIZES)), run(len(ns))
    m = off[len(SIZES)]
    assert np.array_equal(few["acc"], many["acc"][:m])
    assert np.array_equal(few["pot"], many["pot"][:m])
