"""Plane-sweep features of a call with large source images: the device memory kept for images stays
bounded (64 MiB, or one view's images where those are larger) whatever the number of views, and the
features equal those of one call per view bit for bit."""
import ctypes as C
import time

import numpy as np
import pytest

from cumulus3d_amd import init_net, pm

pytestmark = pytest.mark.gpu


def _free(be):
    """Free device memory, through the runtime that the engine itself uses, once earlier frees are through."""
    seen = []
    while len(seen) < 40 and (len(seen) < 4 or len(set(seen[-4:])) > 1):
        free, total = C.c_size_t(), C.c_size_t()
        assert be.L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        seen.append(free.value)
        time.sleep(0.05)
    return seen[-1]


def test_images_of_a_features_call_stay_bounded():
    rng = np.random.default_rng(3)
    keep, views = [], []
    for i in range(6):
        src = [(rng.integers(0, 256, (4000, 4000), dtype=np.uint8), [60.0, 60.0, 2000.0, 2000.0], np.eye(3, dtype=np.float32).ravel(),
                [0.1 * i + 0.2 * j, 0.0, 0.0]) for j in range(2)]
        views.append(init_net.sweep_view(rng.integers(0, 256, (60 - i, 64), dtype=np.uint8), [60.0, 60.0, 32.0, 30.0], src, 2.0, 9.0, keep))
    be = pm.HipPatchMatch()
    one, net = (init_net.InitNet(be, n, 64, 64) for n in (1, 6))
    before = _free(be)
    net.features(0, views)
    taken = before - _free(be)
    for i, v in enumerate(views):
        one.features(0, [v])
        assert np.array_equal(one.get_features(0), net.get_features(i)), i
    be.close()
    assert taken <= (64 << 20) + (4 << 20), taken  # 192 MB of images
