"""Reprojections that leave the float range: IEEE division gives infinity, which the read-out filter
rejects. Counts equal the oracle's."""
import numpy as np
import pytest

from cumulus3d_amd import abi, pm

pytestmark = pytest.mark.gpu


def _right_angle_input():
    """Two views at right angles: the source looks along the reference's x axis, so that a source depth
    moves its point along the reference's x axis and leaves its depth there as it is."""
    w, h = 64, 48
    rng = np.random.default_rng(5)
    k = [50.0, 50.0, 32.0, 24.0]
    r = np.float32([[0, 0, -1], [0, 1, 0], [1, 0, 0]])
    c = np.float32([-10, 0, 10])  # the source's centre, in front of the points at depth 10
    there = (r.ravel(), -r @ c, c)
    back = (r.T.ravel(), c, -r @ c)
    views = [abi.ViewData(key=v + 1, levels=[abi.LevelData(rng.integers(0, 256, (h, w), dtype=np.uint8), k)], sources=[1 - v],
                          pairs=[there if v == 0 else back], depth_min=5.0, depth_max=20.0, k=k) for v in (0, 1)]
    # every window cost and angle passes: the reprojection error alone decides
    return abi.KernelInput(views, abi.fast_profile()[0], abi.FilterParams(min_ncc=-1.0, min_triangulation_angle_deg=0.0, geom_max_cost=1e6))


def test_overflowed_reprojections_are_rejected():
    import oracle

    inp = _right_angle_input()
    st = abi.ViewState(64, 48)
    st.depth[...] = 10.0
    st.normal[...] = np.float32([-0.70710677, 0, -0.70710677])
    orc = oracle.Oracle(inp, threads=4)
    be = pm.HipPatchMatch()
    with be.begin(inp) as s:
        # finite errors; a finite quotient whose square overflows; an infinite product
        for i, (depth, counted) in enumerate([(10.0, True), (1e30, False), (3e37, False), (3e38, False)]):
            snap = abi.DepthSnapshot(i + 1, 0, [None, np.full((48, 64), depth, np.float32)])
            ref = orc.filter([0], [st], snap)[0]
            assert bool(ref.any()) == counted
            assert np.array_equal(s.filter([0], [st], snap)[0], ref), depth
    be.close()
