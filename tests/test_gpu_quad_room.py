"""The second form of the quad table is made only where it leaves the device room for everything else
a session may need; without it every launch samples the 4-byte entries. $C3D_PM_FREE_BYTES stands in
for the device's free memory."""
import ctypes as C
import time

import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu

SRC3 = [[1, 2], [0, 2], [0, 1]]


def _table_bytes(sizes):
    return 8 * sum((((w + 3) * (h + 3)) + 63) // 64 * 64 for w, h in sizes)


def _free(be):
    """Free device memory, through the runtime that the engine itself uses, once earlier frees are through."""
    seen = []
    while len(seen) < 40 and (len(seen) < 4 or len(set(seen[-4:])) > 1):
        free, total = C.c_size_t(), C.c_size_t()
        assert be.L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        seen.append(free.value)
        time.sleep(0.05)
    return seen[-1]


def test_second_table_leaves_room(monkeypatch):
    sizes = [(2000, 1500)] * 3
    sc = scenes.make_mixed_scene(scenes.oblique_rig(3), sizes, seed=3, device=True)
    pmp, fl = abi.fast_profile()
    inp = scenes.kernel_input(sc, SRC3, [(15.0, 120.0)] * 3, pmp, fl)
    need = _table_bytes(sizes)
    be = pm.HipPatchMatch()
    be.begin(inp).close()
    taken = []
    for free in (31 * need, 33 * need):
        monkeypatch.setenv("C3D_PM_FREE_BYTES", str(free))
        before = _free(be)
        with be.begin(inp):
            taken.append(before - _free(be))
    be.close()
    assert taken[1] - taken[0] >= need // 2, (taken, need)


@pytest.mark.parametrize("free", [None, "0"])  # both forms of the table
@pytest.mark.parametrize("window", [(5, 2), (5, 1), (4, 2)])  # held weights, weights formed again, and the any-radius kernels
def test_every_sampling_kernel_in_both_forms(monkeypatch, free, window):
    """Half steps from given planes, evaluation, read-out filter and cost probe against the oracle, over
    views of about a round of 512 tiles (8 XCDs x runs of 64): photometric and geometric."""
    import oracle

    sizes = [(512, 128), (496, 128), (528, 136)]
    sc = scenes.make_mixed_scene(scenes.oblique_rig(3), sizes, seed=37)
    pmp, fl = abi.fast_profile()
    pmp.window_radius, pmp.window_step = window
    inp = scenes.kernel_input(sc, SRC3, [(15.0, 120.0)] * 3, pmp, fl)
    rng = np.random.default_rng(1)
    xy = np.stack([rng.integers(0, 512, 64), rng.integers(0, 128, 64)], 1).astype(np.int32)
    planes = np.concatenate([rng.normal(0, 0.2, (64, 2)), -np.ones((64, 1)), rng.uniform(30, 60, (64, 1))], 1).astype(np.float32)

    def run(engine, pair_costs):
        rng = np.random.default_rng(2)
        st = [abi.ViewState(w, h) for w, h in sizes]
        for q, gd, gn in zip(st, sc.gt_depth, sc.gt_normal):
            q.depth[...] = gd * rng.uniform(0.9, 1.1, gd.shape)
            q.normal[...] = gn
        engine.run([0, 1, 2], st, abi.run_params(0, False, False, 1, 1, False))
        snap = abi.DepthSnapshot(5, 0, [x.depth.copy() for x in st])
        out = engine.evaluate(0, [0, 1, 2], st) + engine.evaluate(0, [0, 1, 2], st, True, snap)
        engine.run([0, 1, 2], st, abi.run_params(0, True, False, 1, 2, False), snap)
        return [x for s in st for x in (s.depth, s.normal, s.cost)] + out + [pair_costs()], engine.filter([0, 1, 2], st, snap)

    o = oracle.Oracle(inp, threads=16)
    ref, rc = run(o, lambda: np.array([o.ncc_cost_f32(0, 0, 0, int(x), int(y), p) for (x, y), p in zip(xy, planes)], np.float32))
    if free is not None:
        monkeypatch.setenv("C3D_PM_FREE_BYTES", free)
    opts = abi.c3d_pm_options()
    opts.any_radius = int(window == (4, 2))
    be = pm.HipPatchMatch(0, opts)
    with be.begin(inp) as s:
        got, gc = run(s, lambda: s.pair_costs(0, 0, 0, xy, planes))
    be.close()
    for a, b in zip(got, ref):
        assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))
    for a, b in zip(gc, rc):
        assert np.array_equal(a, b)
