"""The work queue of the ensemble's persistent kernel is empty again after each
launch (needs an MI355X): repeated launches on few workgroups, on the paths that
take that kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tpt,far", [(2, 0), (4, 0), (1, 3), (1, 4)])
def test_queue_reused_across_launches(pkg, orc, tpt, far):
    ens = pkg.ics.cluster_ensemble(nsys=8, seed=5, nmin=200, nmax=3000)
    off = ens["offsets"]
    runs = []
    with pkg.Ensemble(off, "split") as e:
        e.set_params(1.0, ens["h"], 1e-3)
        e.upload(ens["pos"], ens["vel"], ens["mass"])
        e.set_tuning(targets_per_thread=tpt, blocks=5, resident=0, sort_interval=0, far_path=far)
        for _ in range(4):     # the queue is reset by the last block of each launch
            e.compute_force()
            runs.append(e.download(pos=False, vel=False)["acc"])
    for r in runs[1:]:
        assert np.array_equal(r, runs[0])
    for s in range(len(off) - 1):
        sl = slice(off[s], off[s + 1])
        ref = orc.compute_force(ens["pos"][sl], ens["mass"][sl], [ens["h"][s]] * 6)
        assert np.median(orc.rel_err(runs[0][sl], ref)) <= 1e-6
