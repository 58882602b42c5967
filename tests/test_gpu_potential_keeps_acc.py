"""A potential leaves the accelerations as they were, on every kernel that can
compute it (needs an MI355X)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 5000])
@pytest.mark.parametrize("mode,tpt,far", [("fp64", 1, 0), ("split", 1, 0), ("split", 2, 0), ("split", 4, 3),
                                          ("split", 1, 1), ("split", 1, 2), ("split", 1, 3), ("split", 1, 4),
                                          ("split_central", 1, 0), ("fp32", 1, 0), ("fp32", 2, 0), ("fp32", 4, 0),
                                          ("fp32", 1, 4)])
@pytest.mark.parametrize("nseg", [1, 8])
def test_potential_keeps_accelerations(pkg, mode, tpt, far, n, nseg):
    pos, vel, mass = pkg.ics.plummer(n, seed=5)
    mark = np.arange(3.0 * n).reshape(n, 3)
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, [0.01] * 6)
        ctx.upload(pos, vel, mass)
        if mode == "split_central":
            ctx.set_central(1)
        ctx.set_tuning(tpt, nseg, 16, far)
        ctx.compute_force()
        ctx.upload_acc(mark)
        ctx.compute_potential(self_term=False)
        d = ctx.download(pos=False, vel=False, acc=True, pot=True)
    assert np.array_equal(d["acc"], mark)
    assert np.all(d["pot"] < 0.0)
