"""Force launches of ensembles of small systems (far path 0, one target per lane):
a workgroup's waves without a source tile make room for the next workgroup, so
a launch of 2800 workgroups costs no more per system than one of 8000 (needs an
MI355X)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _force_time(pkg, nsys, n):
    off = np.arange(nsys + 1, dtype=np.int64) * n
    pos, vel, mass = pkg.ics.plummer(nsys * n, seed=3)
    with pkg.Ensemble(off, "split") as e:
        e.set_params(1.0, 0.01, 1e-6)
        e.upload(pos, vel, mass * nsys)
        e.set_tuning(targets_per_thread=1, resident=0, far_path=0)
        t = []
        for _ in range(12):
            a = time.perf_counter()
            for _ in range(10):
                e.compute_force()
            e.sync()
            t.append((time.perf_counter() - a) / 10)
    return min(t)


def test_fewer_systems_take_no_longer_each(pkg):
    few, many = _force_time(pkg, 700, 256), _force_time(pkg, 2000, 256)
    # 0.35 by the systems alone, and a launch's fixed cost; with the idle waves of
    # eight held at the barrier 0.74
    assert few < 0.6 * many, (few, many)
