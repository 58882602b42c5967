"""Results that reach the host in pinned pieces of 2^17 doubles, eight in flight,
by several threads from eight on (needs an MI355X): whole arrays, on the edges
of a piece and of the slots, several downloads at a time.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE = 1 << 17   # doubles


def _state(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((n, 3)), rng.standard_normal((n, 3)), rng.uniform(0.5, 1.0, n)


@pytest.mark.parametrize("n", [1, 255, PIECE // 3, PIECE // 3 + 1, 8 * PIECE // 3 + 1, 400003])
def test_download_returns_the_state(pkg, n):
    pos, vel, mass = _state(n, n)
    acc = np.arange(3.0 * n).reshape(n, 3)
    pot = -np.arange(1.0 * n)
    with pkg._native.Context(n, pkg._native.MODES["fp64"]) as ctx:
        ctx.upload(pos, vel, mass)
        ctx.upload_acc(acc, pot)
        for _ in range(2):
            d = ctx.download(pos=True, vel=True, acc=True, pot=True)
            for key, want in (("pos", pos), ("vel", vel), ("acc", acc), ("pot", pot)):
                assert np.array_equal(d[key], want), key
        assert np.array_equal(ctx.download(pos=False, vel=False, acc=False, pot=True)["pot"], pot)


def test_downloads_from_several_threads(pkg):
    states = [_state(n, n) for n in (700, 60001, 200001, 390001)]
    bad = []

    def work(pos, vel, mass):
        with pkg._native.Context(len(mass), pkg._native.MODES["fp64"]) as ctx:
            ctx.upload(pos, vel, mass)
            for _ in range(3):
                d = ctx.download(pos=True, vel=True, acc=False)
                if not (np.array_equal(d["pos"], pos) and np.array_equal(d["vel"], vel)):
                    bad.append(len(mass))

    threads = [threading.Thread(target=work, args=s) for s in states]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
