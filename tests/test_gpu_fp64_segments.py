"""FP64 forces and potentials of few particles, whose sources are cut at 64
instead of 256, where segments and waves' parts of them end raggedly: a context
and the allocation-free call against the oracle (needs an MI355X).

Tolerance: a sum of n terms in FP64 is within a few n eps of the sum of its
terms' magnitudes; 1e-12 of the largest force is above that up to 4000 terms.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 257, 1000, 2049, 4000])
def test_fp64_forces_of_few_particles(pkg, orc, n):
    torch = pytest.importorskip("torch")
    nat = pkg._native
    pos, vel, mass = pkg.ics.plummer(n, seed=n)
    h = [0.05] * 6
    ref, pref = orc.compute_force(pos, mass, h), orc.compute_potential(pos, mass, h)
    with nat.Context(n, nat.MODES["fp64"]) as ctx:
        ctx.set_params(1.0, h)
        ctx.upload(pos, vel, mass)
        ctx.compute_force()
        ctx.compute_potential(self_term=False)
        d = ctx.download(pos=False, vel=False, acc=True, pot=True)
    x = torch.from_numpy(np.ascontiguousarray(pos.T)).cuda()
    m = torch.from_numpy(mass).cuda()
    out = torch.empty((4, n), dtype=torch.float64, device="cuda")
    p = [out[k].data_ptr() for k in range(4)]
    nat.compute_force_noalloc(nat.MODES["fp64"], n, x[0].data_ptr(), x[1].data_ptr(), x[2].data_ptr(), m.data_ptr(),
                              p[0], p[1], p[2], p[3], h_const=0.05,
                              stream=torch.cuda.current_stream().cuda_stream)
    out = out.cpu().numpy()
    tol, ptol = 1e-12 * max(np.abs(ref).max(), 1.0), 1e-12 * max(np.abs(pref).max(), 1.0)
    for acc, pot in ((d["acc"], d["pot"]), (out[:3].T, out[3])):
        assert np.max(np.abs(acc - ref)) <= tol
        assert np.max(np.abs(pot - pref)) <= ptol
