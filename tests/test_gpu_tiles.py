"""Sizes at the edges of the half step's pixel blocks (16 x 8 pixels a wave with one lane per pixel)
and of the runs of 16 or 64 tiles that are dealt to the 8 XCDs (128 or 512 tiles a round): the engine equals the
oracle bit for bit under every workgroup shape."""
import numpy as np
import pytest

from cumulus3d_amd import abi, pm, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [(16, 8), (15, 7), (17, 9)],          # one block, one pixel less, one more
    [(31, 33), (8, 64), (240, 8)],        # remainders in both directions, one block high
    [(256, 64), (240, 64), (257, 64)],    # 128, 120 and 136 blocks: a whole round, under it, over it
    [(161, 119)] * 3,                     # with no shape asked for: four lanes per pixel (eight above)
    [(255, 161)] * 3,                     # two lanes per pixel
])
def test_block_edges_bit_exact(sizes):
    import oracle

    sc = scenes.make_mixed_scene(scenes.oblique_rig(3), sizes, seed=21)
    pmp, fl = abi.fast_profile()
    inp = scenes.kernel_input(sc, [[1, 2], [0, 2], [0, 1]], [(15.0, 120.0)] * 3, pmp, fl)

    def run(engine):
        st = [abi.ViewState(w, h) for w, h in sizes]
        engine.run([0, 1, 2], st, abi.run_params(0, False, True, 1, 1, False))
        snap = abi.DepthSnapshot(5, 0, [x.depth.copy() for x in st])
        engine.run([0, 1, 2], st, abi.run_params(0, True, False, 1, 2, False), snap)
        return st, engine.filter([0, 1, 2], st, snap)

    ref, rc = run(oracle.Oracle(inp, threads=16))
    for rows, tpp in [(0, 0)] + list(abi.TILE_SHAPES):
        opts = abi.c3d_pm_options()
        opts.tile_rows, opts.threads_per_pixel = rows, tpp
        be = pm.HipPatchMatch(0, opts)
        with be.begin(inp) as s:
            got, gc = run(s)
        be.close()
        for a, b in zip(got, ref):
            for x, y in ((a.depth, b.depth), (a.normal, b.normal), (a.cost, b.cost)):
                assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32)), (rows, tpp)
        for a, b in zip(gc, rc):
            assert np.array_equal(a, b), (rows, tpp)


@pytest.mark.parametrize("width", [1008, 1024, 1040])  # two views: 8064, 8192 and 8320 waves
def test_builds_agree_across_the_geometric_wave_count(width):
    """One-row workgroups take the two-wave build of the half step up to 8192 waves of a geometric run and
    the three-wave build above; two-row workgroups always take the latter. Same states."""
    sizes = [(width, 512)] * 2
    sc = scenes.make_mixed_scene(scenes.oblique_rig(2), sizes, seed=29)
    pmp, fl = abi.fast_profile()
    inp = scenes.kernel_input(sc, [[1], [0]], [(15.0, 120.0)] * 2, pmp, fl)
    outs = []
    for rows in (1, 2):
        opts = abi.c3d_pm_options()
        opts.tile_rows, opts.threads_per_pixel = rows, 1
        be = pm.HipPatchMatch(0, opts)
        with be.begin(inp) as s:
            st = [abi.ViewState(w, h) for w, h in sizes]
            s.run([0, 1], st, abi.run_params(0, False, True, 1, 1, False))
            snap = abi.DepthSnapshot(5, 0, [x.depth.copy() for x in st])
            s.run([0, 1], st, abi.run_params(0, True, False, 1, 2, False), snap)
            outs.append(st)
        be.close()
    for a, b in zip(*outs):
        for x, y in ((a.depth, b.depth), (a.normal, b.normal), (a.cost, b.cost)):
            assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))


@pytest.mark.parametrize("sizes", [
    [(512, 128), (496, 128), (528, 136)],  # 512 tiles (a whole round of runs of 64), fewer, more
    [(130, 200), (17, 300), (300, 17)],    # bands of 8 rows of blocks with a rest, one column, under one band
])
def test_bands_of_blocks_bit_exact(sizes):
    import oracle

    sc = scenes.make_mixed_scene(scenes.oblique_rig(3), sizes, seed=37)
    pmp, fl = abi.fast_profile()
    inp = scenes.kernel_input(sc, [[1, 2], [0, 2], [0, 1]], [(15.0, 120.0)] * 3, pmp, fl)

    def run(engine):
        st = [abi.ViewState(w, h) for w, h in sizes]
        engine.run([0, 1, 2], st, abi.run_params(0, False, True, 2, 1, False))
        return [x for s in st for x in (s.depth, s.normal, s.cost)]

    ref = run(oracle.Oracle(inp, threads=16))
    for rows, tpp in [(0, 0)] + list(abi.TILE_SHAPES):
        opts = abi.c3d_pm_options()
        opts.tile_rows, opts.threads_per_pixel = rows, tpp
        be = pm.HipPatchMatch(0, opts)
        with be.begin(inp) as s:
            got = run(s)
        be.close()
        for a, b in zip(got, ref):
            assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32)), (rows, tpp)
