"""A large download after steps that are still running waits for them with one
thread, as a stream synchronisation does: the threads that empty its pieces
start when there is a piece (needs an MI355X).
"""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_download_waits_with_one_thread(pkg):
    n, steps = 300000, 20      # two arrays of seven pieces; about 20 ms a step
    pos, vel, mass = pkg.ics.plummer(n, seed=5)
    with pkg._native.Context(n, pkg._native.MODES["split"]) as ctx:
        ctx.set_params(1.0, [0.01] * 6)
        ctx.upload(pos, vel, mass)
        ctx.compute_force()
        ctx.download(acc=False)
        wall, cpu = time.perf_counter(), time.process_time()
        ctx.kdk_steps(steps, 1e-6)
        ctx.download(acc=False)
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.05          # the steps, not the copies
    assert cpu < 2.0 * wall, (cpu, wall)
