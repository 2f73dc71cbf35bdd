"""The tile autotuner against the default, which takes two, four or eight lanes per pixel in small
launches: a tuned session is no slower in the launches it was tuned on, nor at the coarse scales of a
job tuned at its top scale. Times are the least of several calls, against a bound of 1.25 (one lane
in place of eight takes more than twice as long)."""
import time

import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu

SRC = [[1, 2], [0, 2], [0, 1]]
SCHEDULE = abi.Schedule(photometric_iters=8, geometric_rounds=0)


def _densify_ms(s, graph):
    tms = [s.densify([0], SCHEDULE)[3] for _ in range(10)]
    return min(t.total_ms if graph else t.half_kernel_ms for t in tms)


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("shape", [(0, 0), (1, 1)])  # untuned, and one lane asked for before tuning
def test_tuning_a_small_job_keeps_its_lanes(graph, shape):
    sc = scenes.make_terrain_scene(scenes.oblique_rig(3), 160, 96, focal=125.0, seed=7)
    pmp, fl = abi.fast_profile()
    inp = scenes.kernel_input(sc, SRC, [(20.0, 80.0)] * 3, pmp, fl)
    ms = []
    for tune in (0, 1):
        opts = abi.c3d_pm_options()
        opts.use_graph = graph
        if tune:
            opts.tile_rows, opts.threads_per_pixel = shape
        be = pm.HipPatchMatch(0, opts)
        with be.begin(inp) as s:
            if tune:
                before = s.densify([0], SCHEDULE)[0][0]  # captured before the shape changes
                chosen = s.autotune([0])
            ms.append(_densify_ms(s, graph))
            after = s.densify([0], SCHEDULE)[0][0]
        be.close()
    for x, y in ((before.depth, after.depth), (before.normal, after.normal), (before.cost, after.cost)):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    print(f"default {ms[0]:.3f} ms, tuned to {chosen[0]} {ms[1]:.3f} ms")
    assert ms[1] <= 1.25 * ms[0]


def test_tuning_the_top_scale_leaves_coarse_scales():
    sc = scenes.make_terrain_scene(scenes.oblique_rig(3), 960, 540, focal=500.0, seed=7)
    pmp, fl = abi.fast_profile()
    be = pm.HipPatchMatch()
    levels = [be.build_pyramid(v.gray, [float(q) for q in v.k], 3) for v in sc.views]
    inp = scenes.kernel_input(sc, SRC, [(20.0, 80.0)] * 3, pmp, fl, levels=levels)
    with be.begin(inp) as s:
        def coarse_ms():
            st, least = abi.ViewState(240, 135), np.inf
            for _ in range(6):
                t = time.perf_counter()
                s.run([0], [st], abi.run_params(0, False, True, 20, 1, False))
                least = min(least, 1e3 * (time.perf_counter() - t))
            return least

        default = coarse_ms()
        chosen = s.autotune([0], level=2)
        tuned = coarse_ms()
    be.close()
    print(f"240 x 135: default {default:.3f} ms, tuned at 960 x 540 to {chosen[0]} {tuned:.3f} ms")
    assert tuned <= 1.25 * default
