"""A missing output array of one view is refused before any work, as C3D_INVALID_ARGUMENT with a message;
the other views' arrays stay untouched and the session stays usable."""
import ctypes as C

import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("missing", [0, 1, 2])
def test_evaluate_and_filter_refuse_a_null_output(missing):
    sc = scenes.make_terrain_scene(scenes.oblique_rig(3), 64, 48, focal=50.0, seed=3)
    pmp, fl = abi.fast_profile()
    inp = scenes.kernel_input(sc, [[1, 2], [0, 2], [0, 1]], [(20.0, 80.0)] * 3, pmp, fl)
    st = [abi.ViewState(64, 48) for _ in range(3)]
    for q, d, n in zip(st, sc.gt_depth, sc.gt_normal):
        q.depth[...], q.normal[...] = d, n
    snap = abi.DepthSnapshot(1, 0, [q.depth for q in st])
    views = abi.views_array([0, 1, 2])
    be = pm.HipPatchMatch()
    with be.begin(inp) as s:
        for dtype, ctype, call in (
            (np.float32, C.c_float, lambda p: s.L.c3d_pm_evaluate(s.h, 0, views, 3, abi.states_array(st), 0, None, p)),
            (np.uint8, C.c_uint8, lambda p: s.L.c3d_pm_filter(s.h, views, 3, abi.states_array(st), C.byref(snap.c), p)),
        ):
            outs = [np.full((48, 64), 77, dtype) for _ in range(3)]
            ptrs = abi.ptr_array(outs, ctype)
            ptrs[missing] = C.POINTER(ctype)()
            assert call(ptrs) == abi.C3D_INVALID_ARGUMENT
            assert "null" in s.L.c3d_pm_last_error().decode()
            assert all((o == 77).all() for o in outs)
            assert call(abi.ptr_array(outs, ctype)) == abi.C3D_OK
            assert not any((o == 77).any() for o in outs)
    be.close()
