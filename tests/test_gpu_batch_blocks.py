"""nb_batch_tuning.blocks bounds the workgroups of the ensemble's force launch on
far path 0 with one target per lane, without a change of its results (needs an
MI355X).
"""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["split", "split_central"])
def test_few_blocks_same_bits(pkg, mode):
    ens = pkg.ics.cluster_ensemble(nsys=24, seed=5, nmin=1, nmax=2000)
    outs, times = [], []
    with pkg.Ensemble(ens["offsets"], mode) as e:
        e.set_params(1.0, ens["h"], 1e-3)
        e.upload(ens["pos"], ens["vel"], ens["mass"])
        if mode == "split_central":
            e.set_central(1)
        for blocks in (0, 2, 37, 1 << 20):
            e.set_tuning(targets_per_thread=1, blocks=blocks, resident=0, sort_interval=0, far_path=0)
            e.compute_force()
            e.compute_potential()
            outs.append(e.download(pos=False, vel=False, acc=True, pot=True))
            t = []
            for _ in range(5):
                a = time.perf_counter()
                e.compute_force()
                e.sync()
                t.append(time.perf_counter() - a)
            times.append(min(t))
    for d in outs[1:]:
        assert all(np.array_equal(d[k], outs[0][k]) for k in d)
    # about 200 workgroups one after the other on two CUs, against one round
    assert times[1] > 5 * times[0], times
