"""Depths at and beyond the ends of the range in which the engine divides by reciprocal and residual
(2^-100 to 2^100; IEEE division outside): costs and a geometric run equal the oracle's bit for bit."""
import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu

SRC3 = [[1, 2], [0, 2], [0, 1]]


def _input(focal=None):
    sc = scenes.make_terrain_scene(scenes.oblique_rig(3), 64, 48, focal=50.0, seed=3)
    if focal:
        for v in sc.views:
            v.k[:2] = focal
    pmp, fl = abi.fast_profile()
    return scenes.kernel_input(sc, SRC3, [(20.0, 80.0)] * 3, pmp, fl)


DEPTHS = np.array([1e-44, 2.0**-101, 2.0**-100, 2.0**-99, 1e-12, 40.0, 2.0**99, 2.0**100, 2.0**101, 2.0**126, 3e38, np.inf], np.float32)


def test_costs_at_extreme_depths():
    import oracle

    inp = _input()
    o = oracle.Oracle(inp, threads=4, rcp_mode=1)
    planes = np.array([[*n, d] for d in DEPTHS for n in ((0, 0, -1), (0, -0.6, -0.8), (0, 0, -1e-20), (0, 0, -1e20))], np.float32)
    xy = np.tile(np.int32([[32, 24]]), (len(planes), 1))
    be = pm.HipPatchMatch()
    with be.begin(inp) as s:
        got = s.pair_costs(0, 0, 0, xy, planes)
    be.close()
    ref = np.array([o.ncc_cost_f32(0, 0, 0, 32, 24, p) for p in planes], np.float32)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("focal", [None, 2.0**-21, 2.0**41])
def test_geometric_run_at_extreme_depths_and_focal_lengths(focal):
    import oracle

    inp = _input(focal)

    def run(engine):
        st = [abi.ViewState(64, 48) for _ in range(3)]
        r = np.random.default_rng(2)
        for q in st:
            q.depth[...] = np.where(r.random(q.depth.shape) < 0.5, r.uniform(20, 80, q.depth.shape), r.choice(DEPTHS[:-1], q.depth.shape))
            q.normal[..., 2] = -1
            q.cost[...] = r.uniform(0, 1, q.cost.shape)
        snap = abi.DepthSnapshot(1, 0, [q.depth.copy() for q in st])
        engine.run([0, 1, 2], st, abi.run_params(0, True, False, 1, 1, False), snap)
        return st, engine.filter([0, 1, 2], st, snap)

    be = pm.HipPatchMatch()
    with be.begin(inp) as s:
        got, gc = run(s)
    be.close()
    ref, rc = run(oracle.Oracle(inp, threads=16))
    for a, b in zip(got, ref):
        for x, y in ((a.depth, b.depth), (a.normal, b.normal), (a.cost, b.cost)):
            assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))
    for a, b in zip(gc, rc):
        assert np.array_equal(a, b)
