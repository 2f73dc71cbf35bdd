"""The window loops that form their weights again: the quality profile's (5, 1), compiled in, and the
any-radius kernels, whose rows are taken in groups of six samples and a rest of one to five. Equal to
the oracle bit for bit, also where the colour sigma makes weights vanish."""
import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma_color", [None, 0.02])
@pytest.mark.parametrize("wr,step,any_radius", [
    (5, 1, 0), (5, 1, 1),                                             # both kernels of the profile's window
    (1, 2, 1), (4, 2, 1),                                             # less than one group: 2 and 5 samples a row
    (5, 2, 1), (6, 2, 0), (7, 2, 0), (8, 2, 0), (9, 2, 0), (10, 2, 0),  # 6 to 11 samples a row
])
def test_recomputed_weights_bit_exact(wr, step, any_radius, sigma_color):
    import oracle

    sizes = [(47, 33), (64, 40), (33, 49)]
    sc = scenes.make_mixed_scene(scenes.oblique_rig(3), sizes, seed=31)
    pmp, fl = abi.fast_profile()
    pmp.window_radius, pmp.window_step = wr, step
    if sigma_color:
        pmp.sigma_color = sigma_color
    inp = scenes.kernel_input(sc, [[1, 2], [0, 2], [0, 1]], [(15.0, 120.0)] * 3, pmp, fl)

    def run(engine):
        st = [abi.ViewState(w, h) for w, h in sizes]
        engine.run([0, 1, 2], st, abi.run_params(0, False, True, 2, 1, False))
        snap = abi.DepthSnapshot(5, 0, [x.depth.copy() for x in st])
        engine.run([0, 1, 2], st, abi.run_params(0, True, False, 1, 2, False), snap)
        return [x for s in st for x in (s.depth, s.normal, s.cost)], engine.filter([0, 1, 2], st, snap)

    ref, rc = run(oracle.Oracle(inp, threads=16))
    opts = abi.c3d_pm_options()
    opts.any_radius = any_radius
    be = pm.HipPatchMatch(0, opts)
    with be.begin(inp) as s:
        got, gc = run(s)
    be.close()
    for a, b in zip(got + list(gc), ref + list(rc)):
        assert np.array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))
