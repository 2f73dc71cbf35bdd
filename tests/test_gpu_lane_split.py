"""Geometric runs whose costs exceed 3 (geom_lambda x geom_max_cost well above 1) with two, four and
eight lanes per pixel: the lanes exchange their refinement candidates' costs, and a candidate that was
given up early must not be accepted whatever the best cost is. Equal to the oracle bit for bit."""
import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(64, 48), (161, 119), (255, 161)])  # eight, four and two lanes with no shape asked for
@pytest.mark.parametrize("any_radius", [0, 1])
def test_costs_above_three_bit_exact(size, any_radius):
    import oracle

    sc = scenes.make_mixed_scene(scenes.oblique_rig(3), [size] * 3, seed=41)
    pmp, fl = abi.fast_profile()
    pmp.geom_lambda = 5.0
    inp = scenes.kernel_input(sc, [[1, 2], [0, 2], [0, 1]], [(15.0, 120.0)] * 3, pmp, fl)

    def run(engine):
        st = [abi.ViewState(*size) for _ in range(3)]
        engine.run([0, 1, 2], st, abi.run_params(0, False, True, 1, 1, False))
        snap = abi.DepthSnapshot(5, 0, [x.depth.copy() for x in st])
        engine.run([0, 1, 2], st, abi.run_params(0, True, False, 2, 2, False), snap)
        return [x for s in st for x in (s.depth, s.normal, s.cost)]

    ref = run(oracle.Oracle(inp, threads=16))
    assert max(float(c.max()) for c in ref[2::3]) > 3.0
    for rows, tpp in [(0, 0), (1, 1), (4, 2)]:
        opts = abi.c3d_pm_options()
        opts.tile_rows, opts.threads_per_pixel, opts.any_radius = rows, tpp, any_radius
        be = pm.HipPatchMatch(0, opts)
        with be.begin(inp) as s:
            got = run(s)
        be.close()
        for a, b in zip(got, ref):
            assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32)), (rows, tpp)
