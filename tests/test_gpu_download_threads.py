"""Downloads of several contexts at a time, each from a host thread of its own: an
error of any of them fails the test (needs an MI355X)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _downloads(pkg, n, repeats):
    rng = np.random.default_rng(n)
    pos, vel = rng.standard_normal((n, 3)), rng.standard_normal((n, 3))
    done = 0
    with pkg._native.Context(n, pkg._native.MODES["fp64"]) as ctx:
        ctx.upload(pos, vel, np.ones(n))
        for _ in range(repeats):
            d = ctx.download(pos=True, vel=True, acc=False)
            assert np.array_equal(d["pos"], pos) and np.array_equal(d["vel"], vel)
            done += 1
    return done


def test_downloads_from_several_threads_report_errors(pkg):
    sizes = (700, 43691, 60001, 200001, 390001, 175000)   # more than the blocks that stay idle
    with ThreadPoolExecutor(len(sizes)) as pool:
        jobs = [pool.submit(_downloads, pkg, n, 5) for n in sizes]
        assert [j.result() for j in jobs] == [5] * len(sizes)
