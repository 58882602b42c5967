"""Force and potential launches that add their own segments' sums (the last
workgroup of 64 targets to arrive): the same bits call after call, and the
oracle's values, where target groups and segments end raggedly (needs an
MI355X).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp64", "split", "fp32", "split_central"])
@pytest.mark.parametrize("n,nseg", [(65, 2), (257, 2), (1000, 5), (4097, 16), (9001, 64)])
def test_sums_repeat_and_match_the_oracle(pkg, orc, mode, n, nseg):
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    if mode == "fp32":
        pos, mass = (v.astype(np.float32).astype(np.float64) for v in (pos, mass))
    h = [0.05] * 6
    with pkg._native.Context(n, pkg._native.MODES[mode]) as ctx:
        ctx.set_params(1.0, h)
        ctx.upload(pos, vel, mass)
        if mode == "split_central":
            ctx.set_central(1)
        ctx.set_tuning(1, nseg, 0, 0)      # no re-sorts: the same sums every time
        runs = []
        for _ in range(3):
            ctx.compute_force()
            ctx.compute_potential(self_term=False)
            runs.append(ctx.download(pos=False, vel=False, acc=True, pot=True))
    for r in runs[1:]:
        assert np.array_equal(r["acc"], runs[0]["acc"]) and np.array_equal(r["pot"], runs[0]["pot"])
    # a lost or doubled segment is off by the order of 1 / segments
    ref, pref = orc.compute_force(pos, mass, h), orc.compute_potential(pos, mass, h)
    tol = 1e-12 if mode == "fp64" else 1e-4
    assert np.max(np.abs(runs[0]["acc"] - ref)) <= tol * np.max(np.abs(ref))
    assert np.max(np.abs(runs[0]["pot"] - pref)) <= tol * np.max(np.abs(pref))
