"""Threads that share one network: features into slots of their own, with images of different sizes, and
predictions of different batches equal those of one thread bit for bit."""
import threading

import numpy as np
import pytest

from cumulus3d_amd import init_net, pm

pytestmark = pytest.mark.gpu

H, W = 64, 96


def _views(rng, n, side, keep):
    views = []
    for i in range(n):
        src = [(rng.integers(0, 256, (side, side + 9 * j), dtype=np.uint8), [60.0, 60.0, side / 2, side / 2],
                np.eye(3, dtype=np.float32).ravel(), [0.2 * i + 0.1 * j - 0.3, 0.0, 0.0]) for j in range(2)]
        views.append(init_net.sweep_view(rng.integers(0, 256, (H - i, W), dtype=np.uint8), [60.0, 60.0, 48.0, 32.0], src, 2.0, 9.0, keep))
    return views


def _together(*jobs):
    errors = []

    def call(job):
        try:
            for _ in range(20):
                job()
        except BaseException as e:  # reported by the test, not by the thread
            errors.append(e)

    threads = [threading.Thread(target=call, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


def test_two_threads_on_one_network():
    rng, keep = np.random.default_rng(4), []
    small, large = _views(rng, 2, 80, keep), _views(rng, 2, 700, keep)
    be = pm.HipPatchMatch()
    alone, net = (init_net.InitNet(be, 4, H, W, seed=5) for _ in range(2))
    alone.features(0, small)
    alone.features(2, large)

    def features(slot, views):
        net.features(slot, views)
        for i in range(2):
            assert np.array_equal(net.get_features(slot + i), alone.get_features(slot + i)), (slot, i)

    _together(lambda: features(0, small), lambda: features(2, large))
    want = {b: alone.predict(b, want_head=True) for b in (1, 4)}

    def predict(b):
        for x, y in zip(net.predict(b, want_head=True), want[b]):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), b

    _together(lambda: predict(1), lambda: predict(4))
    be.close()
