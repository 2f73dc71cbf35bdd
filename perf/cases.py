"""The work that users have this framework do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" is one use of a public entry point:

  learned   images to read-out depth maps through the learned initialiser (begin, densify_learned)
  fast      images to read-out depth maps by the multi-scale fast profile (build_pyramid, begin,
            densify with post-processing)
  run       one PatchStereo run of a session over caller-held states (photometric or geometric)
  readout   the read-out calls on caller-held states (evaluate, median_filter, filter)
  post      speckle removal and hole filling of one depth map
  fuse      agreement fusion of depth maps into a point cloud
  scene     source views and depth ranges from sparse tracks
  predict   plane-sweep features and the network's prediction for a batch of views
  train     one training step of the network: labels in, losses and gradients out

Scenes are the repository's rendered terrain, seen by formation flights with the benchmark's
intrinsics, noise and depth range. The calls take and return host arrays, so a pass goes from host
memory to host memory.
"""
from __future__ import annotations

import math
import os
from types import SimpleNamespace

import numpy as np
import torch

from cumulus3d_amd import abi, fusion, init_net, neighbors, pm, scenes

NEAR, FAR = 15.0, 120.0  # depth range of the terrain flights, metres
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(init_net.__file__)), "weights", "init_unet.npy")

# ---------------------------------------------------------------- the cases


def listed():
    return [
        # a flight's strip at camera resolution, one job from images to results: the headline path
        dict(name="learned_1080p", kind="learned", width=1920, height=1080, views=9, sources=6, refine=1, geo=1),
        # the fast profile's whole multi-scale schedule at its usual 960-pixel size, many sources
        dict(name="fast_960x540", kind="fast", width=960, height=540, views=12, sources=9),
        # the smallest job: a thumbnail pair preview, where launches and transfers count
        dict(name="run_small", kind="run", width=160, height=96, views=3, run=1, sources=2, iters=2, geometric=False,
             radius=5, step=2, mixed=False),
        # plain estimation from a random start at camera resolution
        dict(name="run_photo_1080p", kind="run", width=1920, height=1080, views=9, run=2, sources=6, iters=3, geometric=False,
             radius=5, step=2, mixed=False),
        # a geometric round over views of several odd sizes in one batch
        dict(name="run_geo_mixed", kind="run", width=1283, height=717, views=9, run=9, sources=5, iters=2, geometric=True,
             radius=5, step=2, mixed=True),
        # the quality profile's window (every pixel of 11 x 11) at a moderate odd size
        dict(name="run_quality", kind="run", width=641, height=479, views=6, run=3, sources=3, iters=2, geometric=False,
             radius=5, step=1, mixed=False),
        # costs, median and consistency counts of finished maps
        dict(name="readout_1080p", kind="readout", width=1920, height=1080, views=9, run=3, sources=6),
        # clean-up of one camera-resolution map
        dict(name="post_1080p", kind="post", width=1920, height=1080),
        # maps of a strip to one cloud
        dict(name="fuse_960x540", kind="fuse", width=960, height=540, views=9, sources=6),
        # scene preparation of a whole zone
        dict(name="scene_108", kind="scene", views=108, points=60000),
        # the initialiser used by itself on a batch of quarter-resolution views
        dict(name="predict_batch", kind="predict", width=480, height=270, batch=6),
        # training on the batch the project trains with
        dict(name="train_batch", kind="train", width=480, height=270, batch=8),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """width and height: widths even over their logarithm, aspects from square to 16:9."""
    w = _log(rng, lo, hi)
    return dict(width=w, height=max(24, int(w * rng.uniform(0.55, 1.0) * (0.75 if w > 1440 else 1.0))))


def _draw(rng):
    kind = rng.choice(["learned", "fast", "run", "run", "run", "readout", "post", "fuse", "scene", "predict", "train"])
    if kind == "learned":
        v = 3 * rng.randint(2, 3)
        return dict(kind=kind, **_size(rng, 320, 1920), views=v, sources=rng.randint(2, v - 3), refine=rng.randint(1, 2), geo=1)
    if kind == "fast":
        v = 3 * rng.randint(2, 4)
        return dict(kind=kind, **_size(rng, 320, 960), views=v, sources=rng.randint(2, v - 3))
    if kind == "run":
        v = 3 * rng.randint(2, 3)
        geometric = rng.random() < 0.5
        radius, step = rng.choice([(5, 2), (5, 2), (5, 2), (4, 2), (3, 1), (5, 1)])
        return dict(kind=kind, **_size(rng, 64, 1920 if step == 2 else 700), views=v, run=rng.randint(1, 3), sources=rng.randint(2, v - 3),
                    iters=rng.randint(1, 3), geometric=geometric, radius=radius, step=step, mixed=rng.random() < 0.3)
    if kind == "readout":
        return dict(kind=kind, **_size(rng, 96, 1920), views=9, run=rng.randint(1, 3), sources=rng.randint(2, 6))
    if kind == "post":
        return dict(kind=kind, **_size(rng, 96, 1920))
    if kind == "fuse":
        return dict(kind=kind, **_size(rng, 96, 960), views=9, sources=rng.randint(4, 6))
    if kind == "scene":
        return dict(kind=kind, views=3 * rng.randint(4, 36), points=_log(rng, 500, 60000))
    return dict(kind=kind, **_size(rng, 64, 480), batch=rng.randint(1, 8))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


# ---------------------------------------------------------------- inputs


def _terrain(case, seed, quarter=False):
    """Rendered terrain views of a formation flight (or three views of one spot), noise included."""
    n = case.get("views", 9)
    w, h = case["width"], case["height"]
    cams = scenes.formation_rig(n // 3, 3) if n > 3 else scenes.oblique_rig(3)
    sizes = [(w, h)] * n
    if case.get("mixed"):
        sizes = [((w * k // 6) | 1, (h * k // 6) | 1) for k in ((6, 4, 3)[i % 3] for i in range(n))]
    sc = scenes.make_mixed_scene(cams, sizes, seed=1000 + seed, noise_sigma=0.01, noise_seed=seed + 1, device=True)
    src = scenes.nearest_sources(sc, [case.get("sources", 2)] * n)
    return sc, src


def _params(case):
    pmp, fl = abi.fast_profile()
    if "radius" in case:
        pmp = abi.PmParams(window_radius=case["radius"], window_step=case["step"])
    return pmp, fl


def _input(sc, src, case, levels=None):
    pmp, fl = _params(case)
    return scenes.kernel_input(sc, src, [(NEAR, FAR)] * len(sc.views), pmp, fl, levels=levels)


def _maps(sc, seed):
    """Depth, normal and cost as a finished run leaves them: the surface with small errors, one
    pixel in twenty wrong, each with the cost that goes with it."""
    rng = np.random.default_rng(seed + 77)
    out = []
    for d0, n0 in zip(sc.gt_depth, sc.gt_normal):
        shape = d0.shape
        d = d0 * (1 + 0.002 * rng.standard_normal(shape, np.float32))
        n = n0 + 0.05 * rng.standard_normal((*shape, 3), np.float32)
        n /= np.maximum(np.linalg.norm(n, axis=-1, keepdims=True), 1e-6)
        cost = np.abs(0.15 * rng.standard_normal(shape, np.float32)) + 0.05
        wrong = rng.random(shape, np.float32) < 0.05
        d = np.where(wrong, NEAR + (FAR - NEAR) * rng.random(shape, np.float32), d)
        d = np.where(d0 > 0, d, 0)
        cost = np.where(wrong, 0.6 + 0.8 * rng.random(shape, np.float32), cost)
        out.append((np.ascontiguousarray(d, np.float32), np.ascontiguousarray(n, np.float32), np.ascontiguousarray(cost, np.float32)))
    return out


def _state(d, n, c):
    s = abi.ViewState(d.shape[1], d.shape[0])
    s.depth, s.normal, s.cost = d.copy(), n.copy(), c.copy()
    return s


def _one_map(case, seed):
    """One depth map before clean-up: speckles (some of low cost, which stay), holes, its raw cost,
    its image and its intrinsics."""
    sc, _ = _terrain(dict(case, views=3), seed)
    rng = np.random.default_rng(seed + 5)
    h, w = sc.gt_depth[0].shape
    d = sc.gt_depth[0] * (1 + 0.002 * rng.standard_normal((h, w), np.float32))
    n = sc.gt_normal[0].copy()
    c = np.abs(0.15 * rng.standard_normal((h, w), np.float32)) + np.float32(0.05)
    for kind in range(3):  # speckles with high cost, speckles with low cost, holes
        for _ in range(max(4, h * w // 8000)):
            r = int(rng.integers(1, max(2, min(h, w) // 60)))
            y, x = int(rng.integers(0, h)), int(rng.integers(0, w))
            sl = (slice(max(0, y - r), y + r + 1), slice(max(0, x - r), x + r + 1))
            if kind == 2:
                d[sl] = 0
            else:
                d[sl] *= 1.3
                c[sl] = (0.7, 0.1)[kind]
    n[d <= 0] = 0
    raw = np.where(d > 0, c, 0.3 + 0.9 * rng.random((h, w), np.float32)).astype(np.float32)
    return d, n, c, raw, sc.views[0].gray, sc.views[0].k


def _tracks(case, seed):
    """Cameras of a formation flight and sparse points with tracks of 2 to 12 views."""
    rng = np.random.default_rng(seed + 11)
    cams = scenes.formation_rig(case["views"] // 3, 3)
    views = []
    for i, (c, t) in enumerate(cams):
        r, tt = scenes.look_at(c, t)
        views.append(scenes.DenseView("v%d" % i, 1920, 1080, np.array([500.0, 500.0, 959.5, 539.5]), r, tt, None))
    ctr = np.array([v.center() for v in views])
    pts = []
    while len(pts) < case["points"]:
        m = case["points"] - len(pts)
        lo, hi = ctr.min(0), ctr.max(0)
        x = np.stack([rng.uniform(lo[0] - 20, hi[0] + 20, m), rng.uniform(lo[1], hi[1] + 50, m), rng.uniform(-8, 8, m)], 1)
        seen = np.zeros((m, len(views)), bool)
        for j, v in enumerate(views):
            q = x @ v.r.T + v.t
            z = np.maximum(q[:, 2], 1e-9)
            u, w = 500 * q[:, 0] / z + 959.5, 500 * q[:, 1] / z + 539.5
            seen[:, j] = (q[:, 2] > 1) & (u >= 0) & (u < 1920) & (w >= 0) & (w < 1080)
        length = 2 + np.minimum(rng.geometric(0.3, m) - 1, 10)
        for p in range(m):
            vis = np.flatnonzero(seen[p])
            if len(vis) >= 2:
                pts.append(scenes.ScenePoint(x[p], [int(k) for k in rng.permutation(vis)[: length[p]]]))
    return scenes.DenseScene(views, pts)


def _net_size(case):
    return -(-case["height"] // 8) * 8, -(-case["width"] // 8) * 8


def _sweep_views(case, seed):
    sc, src = _terrain(dict(case, views=9, sources=2), seed)
    out = []
    for v in range(case["batch"]):
        g = [(sc.views[s].gray, sc.views[s].k, *scenes.pair_geometry(sc, v, s)[:2]) for s in src[v]]
        out.append((sc.views[v].gray, sc.views[v].k, g))
    return sc, out


def _labels(sc, case, b):
    """Depth and normals of the pixels that carry a label, padded to the network's size."""
    hh, ww = _net_size(case)
    d, n = np.zeros((hh, ww), np.float32), np.zeros((hh, ww, 3), np.float32)
    h, w = case["height"], case["width"]
    d[:h, :w], n[:h, :w] = sc.gt_depth[b], sc.gt_normal[b]
    return d, n


# What a program keeps between jobs: the device handle and a loaded network.
_kept = {}


def _backend():
    if "backend" not in _kept:
        _kept["backend"] = pm.HipPatchMatch(0)
    return _kept["backend"]


def _weights():
    return np.load(WEIGHTS, allow_pickle=False).astype(np.float32)


def _network(batch, h, w):
    key = (batch, h, w)
    if _kept.get("net_key") != key:
        if "net" in _kept:
            _kept.pop("net").close()
        net = init_net.InitNet(_backend(), batch, h, w)
        net.set_params(_weights())
        _kept["net"], _kept["net_key"] = net, key
    return _kept["net"]


def prepare(case, seed):
    s = SimpleNamespace(case=case, kind=case["kind"])
    kind = s.kind
    if kind in ("learned", "fast"):
        s.be = _backend()
        s.sc, s.src = _terrain(case, seed)
        s.views = list(range(case["views"]))
    if kind == "learned":
        s.inp = _input(s.sc, s.src, case)
        s.net = _network(8, -(-(case["height"] // 4) // 8) * 8, -(-(case["width"] // 4) // 8) * 8)
        s.schedule = init_net.LearnedSchedule(refine_iters=case["refine"], geometric_rounds=case["geo"], geometric_iters=1, conf_min=0.0)
        s.out = init_net.output_buffers(s.inp, s.views)
    elif kind == "fast":
        s.levels = pm.num_levels(min(case["width"], case["height"]), 3, 64)
        s.schedule = abi.Schedule(post=abi.PostParams.fast())
    elif kind in ("run", "readout"):
        # a backend has one open session at a time, so every held session has its own
        sc, src = _terrain(case, seed)
        s.be = pm.HipPatchMatch(0)
        s.session = s.be.begin(_input(sc, src, case))
        s.views = list(range(case["run"]))
        maps = _maps(sc, seed)
        s.maps = [m[0] for m in maps]
        s.round = 0
        if kind == "run" and not case["geometric"]:
            s.states = [abi.ViewState(sc.views[v].width, sc.views[v].height) for v in s.views]
        else:
            s.states = [_state(*maps[v]) for v in s.views]
    elif kind == "post":
        s.be = _backend()
        s.map = _one_map(case, seed)
        s.params = abi.PostParams.fast()
    elif kind == "fuse":
        s.be = _backend()
        sc, src = _terrain(case, seed)
        maps = _maps(sc, seed)
        s.keep = []
        s.arr = fusion.fusion_views(sc, [m[0] for m in maps], [m[1] for m in maps], [m[2] for m in maps], src, src, s.keep)
        s.capacity = sum(m[0].size for m in maps)
        s.params = fusion.FusionParams()
    elif kind == "scene":
        s.be = _backend()
        s.sparse = neighbors.SparseScene(_tracks(case, seed))
    else:
        s.be = _backend()
        sc, views = _sweep_views(case, seed)
        s.keep = []
        s.views = [init_net.sweep_view(g, k, src, NEAR, FAR, s.keep) for g, k, src in views]
        h, w = _net_size(case)
        if kind == "predict":
            s.net = _network(case["batch"], h, w)
        else:
            s.net = init_net.InitNet(s.be, case["batch"], h, w)
            s.net.set_params(_weights())
            s.net.features(0, s.views)
            s.labels = [_labels(sc, case, b) for b in range(case["batch"])]
            # the smallest rate of a decayed schedule: repeated steps stay at the same point
            s.train = init_net.TrainParams(lr=1e-6)
    return s


# ---------------------------------------------------------------- one pass


def _planes(states):
    return [[q.depth, q.normal, q.cost] for q in states]


def run(s):
    case = s.case
    if s.kind == "learned":
        with s.be.begin(s.inp) as session:
            states, counts, raw, *_ = init_net.densify_learned(session, s.net, s.views, s.schedule, out=s.out)
        return _planes(states), counts, raw
    if s.kind == "fast":
        levels = [s.be.build_pyramid(v.gray, v.k, s.levels) for v in s.sc.views]
        with s.be.begin(_input(s.sc, s.src, case, levels)) as session:
            states, counts, raw, _ = session.densify(s.views, s.schedule)
        return _planes(states), counts, raw
    if s.kind == "run":
        s.round += 1
        snap = abi.DepthSnapshot(s.round, 0, s.maps) if case["geometric"] else None
        p = abi.run_params(0, case["geometric"], not case["geometric"], case["iters"], 1, False)
        s.session.run(s.views, s.states, p, snap)
        return _planes(s.states)
    if s.kind == "readout":
        s.round += 1
        costs = s.session.evaluate(0, s.views, s.states)
        smooth = s.session.median_filter(0, s.views, s.states)
        counts = s.session.filter(s.views, smooth, abi.DepthSnapshot(s.round, 0, s.maps))
        return costs, [[q.depth, q.normal] for q in smooth], counts
    if s.kind == "post":
        d, n, c, raw, gray, k = s.map
        d, n, c = d.copy(), n.copy(), c.copy()  # cleaned in place: the caller keeps its own
        removed = s.be.remove_speckles(d, n, c, s.params)
        filled = s.be.fill_holes(d, n, c, raw, gray, k, s.params)
        return d, n, c, removed, filled
    if s.kind == "fuse":
        cloud = fusion.fuse(s.be, s.arr, s.params, s.capacity)
        # the caller's whole buffers (of the capacity asked for), of which the cloud is the first part
        return cloud.positions.base, cloud.normals.base, cloud.colors.base, cloud.keys.base.view(np.int64), len(cloud.keys)
    if s.kind == "scene":
        count, q75 = neighbors.pair_stats(s.be, s.sparse)
        chosen = neighbors.select_all(count, q75)
        sources = np.full((len(chosen), 10), -1, np.int64)
        for v, c in enumerate(chosen):
            sources[v, : len(c)] = c
        ranges = neighbors.depth_ranges(s.be, s.sparse)
        return count, q75, sources, np.array([r or (0.0, 0.0) for r in ranges])
    if s.kind == "predict":
        s.net.features(0, s.views)
        return s.net.predict(case["batch"], want_head=True)
    for b, (d, n) in enumerate(s.labels):
        s.net.set_labels(b, d, n, case["width"], case["height"], NEAR, FAR)
    return s.net.train_step(case["batch"], s.train, step=True, want_grads=True)


# ---------------------------------------------------------------- what a pass cannot do without

SAMPLE_FLOPS = 28  # one bilinear source sample of a matching window: projection, divide, lerp, sums


def _pixels(case, n):
    if case.get("mixed"):
        f = [(6, 4, 3)[i % 3] for i in range(n)]
        return sum(((case["width"] * k // 6) | 1) * ((case["height"] * k // 6) | 1) for k in f)
    return case["width"] * case["height"] * n


def _net_flops(case):
    px = case["batch"] * _net_size(case)[0] * _net_size(case)[1]
    return 2.0 * px * sum(cin * cout * k * k / 4 ** lv for cin, cout, k, lv in _LAYERS)


def work(case):
    kind = case["kind"]
    if kind in ("learned", "fast", "run", "readout"):
        r, st = case.get("radius", 5), case.get("step", 2)
        window = ((2 * r) // st + 1) ** 2
        px = _pixels(case, case.get("run", case["views"]))
        scale = 1.0
        if kind == "learned":
            per = 15 * (case["refine"] + case["geo"]) + 1  # 9 propagated + 6 refined planes an iteration, one read-out
        elif kind == "fast":
            per, scale = 15 * 7 + 1, 1 + (10 / 7) / 4 + (10 / 7) / 16  # 3 + 2 x 2 iterations, 6 + 2 x 2 on the coarsest scale
        elif kind == "run":
            per = 15 * case["iters"]
        else:
            per = 2
        images = _pixels(case, case["views"]) if kind in ("learned", "fast") else 0
        given = 0 if kind in ("learned", "fast") or (kind == "run" and not case["geometric"]) else 20 * px
        given += 4 * _pixels(case, case["views"]) if kind == "readout" or case.get("geometric") else 0
        wrote = {"learned": 25, "fast": 25, "run": 20, "readout": 21}[kind] * px
        return {"bytes": images + given + wrote, "flops": float(SAMPLE_FLOPS) * window * per * case["sources"] * px * scale}
    if kind == "post":
        px = case["width"] * case["height"]
        return {"bytes": px * (20 + 5 + 20), "flops": px * 20.0}
    if kind == "fuse":
        px = _pixels(case, case["views"])
        return {"bytes": px * (21 + 35 / case["sources"]), "flops": px * 100.0 * case["sources"] / 2}
    if kind == "scene":
        obs = case["points"] * 4.3
        return {"bytes": case["points"] * 32 + obs * 4 + case["views"] ** 2 * 12, "flops": obs * 200.0}
    px = case["batch"] * _net_size(case)[0] * _net_size(case)[1]
    if kind == "predict":
        return {"bytes": px * (3 + 40) + 2.1e6, "flops": _net_flops(case) + px * 64 * 30.0}
    return {"bytes": px * (16 + 128) + 20e6, "flops": 3 * _net_flops(case)}


# ---------------------------------------------------------------- the same in 64 bits

F = torch.float64


def _t(a):
    t = torch.from_numpy(np.ascontiguousarray(a))
    t = t.to("cuda") if torch.cuda.is_available() else t
    return t.to(F) if t.is_floating_point() or t.dtype == torch.uint8 else t


def _np(t):
    return t.detach().cpu().numpy()


def _rays(k, h, w, dev):
    y, x = torch.meshgrid(torch.arange(h, dtype=F, device=dev), torch.arange(w, dtype=F, device=dev), indexing="ij")
    return torch.stack([(x - k[2]) / k[0], (y - k[3]) / k[1], torch.ones_like(x)], -1), x, y


def _shift(img, dy, dx, fill=0.0):
    """img[y + dy, x + dx], `fill` outside."""
    h, w = img.shape[:2]
    out = torch.full_like(img, fill)
    y0, y1, x0, x1 = max(0, -dy), min(h, h - dy), max(0, -dx), min(w, w - dx)
    if y0 < y1 and x0 < x1:
        out[y0:y1, x0:x1] = img[y0 + dy : y1 + dy, x0 + dx : x1 + dx]
    return out


def _bilinear(img, u, v):
    """Bilinear samples of img, 0 outside."""
    h, w = img.shape
    x0, y0 = torch.floor(u).clamp(-2, w), torch.floor(v).clamp(-2, h)
    ax, ay = u - torch.floor(u), v - torch.floor(v)

    def at(x, y):
        ok = (x >= 0) & (y >= 0) & (x < w) & (y < h)
        return torch.where(ok, img[y.clamp(0, h - 1).long(), x.clamp(0, w - 1).long()], 0.0)

    top = at(x0, y0) * (1 - ax) + at(x0 + 1, y0) * ax
    bot = at(x0, y0 + 1) * (1 - ax) + at(x0 + 1, y0 + 1) * ax
    return top * (1 - ay) + bot * ay


def _window_costs(sc, src, v, depth, normal, pmp):
    """Top-K mean over the sources of 1 - bilateral NCC of every pixel's plane."""
    ref = sc.views[v]
    img = _t(ref.gray)
    h, w = img.shape
    ray, _, _ = _rays(ref.k, h, w, img.device)
    off = [(dy, dx) for dy in range(-pmp.window_radius, pmp.window_radius + 1, pmp.window_step)
           for dx in range(-pmp.window_radius, pmp.window_radius + 1, pmp.window_step)]
    s2, c2 = 2 * pmp.sigma_s() ** 2, 2 * (255 * pmp.sigma_color) ** 2
    wgt, sw, mu = [], 0.0, 0.0
    for dy, dx in off:
        i = _shift(img, dy, dx)
        wgt.append(torch.exp(-(dx * dx + dy * dy) / s2 - (img - i) ** 2 / c2))
        sw, mu = sw + wgt[-1], mu + wgt[-1] * i
    mu = mu / sw
    var = sum(g * (_shift(img, dy, dx) - mu) ** 2 for g, (dy, dx) in zip(wgt, off)) / sw
    least = 1e-5 * 65025.0
    facing = (normal * ray).sum(-1)
    c = depth * facing  # n . X of the plane
    costs = []
    for j in src[v]:
        r9, t3, _ = scenes.pair_geometry(sc, v, j)
        rot, tr, ks = _t(r9.reshape(3, 3)), _t(t3), sc.views[j].k
        other = _t(sc.views[j].gray)

        def project(dy, dx):
            q = ray + torch.tensor([dx / ref.k[0], dy / ref.k[1], 0.0], dtype=F, device=img.device)
            # the ray's point on the plane up to the factor n . q, which has the sign of c in front
            p = q @ rot.T + tr * ((normal * q).sum(-1) / c)[..., None]
            return ks[0] * p[..., 0] / p[..., 2] + ks[2], ks[1] * p[..., 1] / p[..., 2] + ks[3], p[..., 2]

        u, q, z = project(0, 0)
        ok = (c < -1e-12) & (z > 1e-8) & (u >= 0) & (q >= 0) & (u <= other.shape[1] - 1) & (q <= other.shape[0] - 1) & (var >= least)
        m = mm = mi = 0.0
        for g, (dy, dx) in zip(wgt, off):
            u, q, z = project(dy, dx)
            sv = torch.where(z > 1e-8, _bilinear(other, torch.nan_to_num(u), torch.nan_to_num(q)), 0.0) - img
            m, mm, mi = m + g * sv, mm + g * sv * sv, mi + g * sv * _shift(img, dy, dx)
        m = m / sw
        vs = mm / sw - m * m
        cc = (1 - (mi / sw - mu * m) / torch.sqrt(var * vs)).clamp(0, 2)
        costs.append(torch.where(ok & (vs >= least), cc, 2.0))
    k = min(pmp.top_k, len(costs))
    best = torch.sort(torch.stack(costs), 0).values[:k].mean(0)
    return torch.where(depth > 0, best, 2.0)


def _median_planes(view, depth, normal):
    """Lower median of the depths that the 5 x 5 neighbours' planes give the pixel, and its normal."""
    h, w = depth.shape
    ray, _, _ = _rays(np.asarray(view.k, np.float32).astype(np.float64), h, w, depth.device)
    rec = torch.where(depth > 0, depth * (normal * ray).sum(-1), torch.nan)
    ds = []
    for dy in range(-2, 3):
        for dx in range(-2, 3):
            den = (_shift(normal, dy, dx) * ray).sum(-1)
            d = _shift(rec, dy, dx, math.nan) / den
            ds.append(torch.where((den < -1e-6) & (d > 0) & torch.isfinite(d), d, torch.inf))
    ds = torch.stack(ds)
    order = torch.sort(ds, dim=0, stable=True)
    cnt = torch.isfinite(ds).sum(0)
    pick = ((cnt - 1).clamp(min=0) // 2)[None]
    d, idx = order.values.gather(0, pick)[0], order.indices.gather(0, pick)[0]
    normals = torch.stack([_shift(normal, dy, dx) for dy in range(-2, 3) for dx in range(-2, 3)])
    n = normals.gather(0, idx[None, ..., None].expand(1, h, w, 3))[0]
    use = (depth > 0) & (cnt > 0)
    return torch.where(use, d, depth), torch.where(use[..., None], n, normal)


def _exact_readout(case, seed):
    sc, src = _terrain(case, seed)
    maps = _maps(sc, seed)
    pmp, _ = _params(case)
    costs, planes = [], []
    for v in range(case["run"]):
        d, n = _t(maps[v][0]), _t(maps[v][1])
        costs.append(_np(_window_costs(sc, src, v, d, n, pmp)))
        md, mn = _median_planes(sc.views[v], d, n)
        planes.append([_np(md), _np(mn)])
    return costs, planes, [None] * case["run"]


def _components(d, rel):
    """Labels of the 4-neighbour components of pixels whose depths join."""
    h, w = d.shape
    label = torch.arange(h * w, device=d.device).reshape(h, w)
    on = d > 0
    right = on[:, :-1] & on[:, 1:] & ((d[:, 1:] - d[:, :-1]).abs() <= rel * torch.minimum(d[:, 1:], d[:, :-1]))
    down = on[:-1] & on[1:] & ((d[1:] - d[:-1]).abs() <= rel * torch.minimum(d[1:], d[:-1]))
    while True:
        new = label.clone()
        lr, ld = torch.minimum(label[:, :-1], label[:, 1:]), torch.minimum(label[:-1], label[1:])
        new[:, :-1] = torch.where(right, torch.minimum(new[:, :-1], lr), new[:, :-1])
        new[:, 1:] = torch.where(right, torch.minimum(new[:, 1:], lr), new[:, 1:])
        new[:-1] = torch.where(down, torch.minimum(new[:-1], ld), new[:-1])
        new[1:] = torch.where(down, torch.minimum(new[1:], ld), new[1:])
        flat = new.reshape(-1)
        root = flat.scatter_reduce(0, label.reshape(-1), flat, "amin")  # a component's label falls with any of its pixels
        new = root[root[flat]].reshape(h, w)
        if torch.equal(new, label):
            return label, on
        label = new


def _exact_post(case, seed):
    d, n, c, raw, gray, k = _one_map(case, seed)
    p = abi.PostParams.fast()
    h, w = d.shape
    d, n, c, raw, gray = _t(d), _t(n), _t(c), _t(raw), _t(gray)
    least = math.ceil(h * w * p.speckle_min_area_frac)
    if least > 1:
        label, on = _components(d, p.speckle_rel_depth)
        order = torch.argsort(c.reshape(-1), stable=True)
        lab = label.reshape(-1)[order]
        by = torch.argsort(lab, stable=True)
        lab, cost = lab[by], c.reshape(-1)[order][by]
        ids, cnt = torch.unique_consecutive(lab, return_counts=True)
        start = torch.cumsum(cnt, 0) - cnt
        gone = (cnt < least) & (cost[start + cnt // 2] > p.speckle_keep_cost)
        erase = torch.zeros(h * w, dtype=torch.bool, device=d.device)
        erase[ids[gone]] = True
        erase = erase[label] & on
        d, n = torch.where(erase, 0.0, d), torch.where(erase[..., None], 0.0, n)
    valid = d > 0
    most = max(1, int(math.floor(math.hypot(w, h) * p.fill_max_frac + 0.5)))
    step = int(np.float32(p.fill_edge_step) * np.float32(255))
    ys, xs = torch.nonzero(~valid & ~(raw > p.fill_max_cost), as_tuple=True)
    ip = gray[ys, xs]
    bd, bs = torch.full_like(ip, math.inf), torch.full_like(ip, math.inf)
    by, bx = torch.zeros_like(ys), torch.zeros_like(xs)
    for ddx, ddy in ((1, 0), (-1, 0), (0, 1), (0, -1), (1, 1), (-1, -1), (1, -1), (-1, 1)):
        prev, going = ip.clone(), torch.ones_like(ys, dtype=torch.bool)
        for q in range(1, most + 1):
            y, x = ys + ddy * q, xs + ddx * q
            going = going & (x >= 0) & (y >= 0) & (x < w) & (y < h)
            yc, xc = y.clamp(0, h - 1), x.clamp(0, w - 1)
            g = gray[yc, xc]
            going = going & ((g - prev).abs() <= step)
            hit = going & valid[yc, xc]
            dd = (g - ip).abs()
            better = hit & ((dd < bd) | ((dd == bd) & (q < bs)))
            bd, bs = torch.where(better, dd, bd), torch.where(better, float(q), bs)
            by, bx = torch.where(better, yc, by), torch.where(better, xc, bx)
            going, prev = going & ~hit, g
    ray, _, _ = _rays(k, h, w, d.device)
    nq = n[by, bx]
    den = (nq * ray[ys, xs]).sum(-1)
    dn = d[by, bx] * (nq * ray[by, bx]).sum(-1) / den
    ok = torch.isfinite(bd) & ~(den > -1e-6) & (dn > 0) & torch.isfinite(dn)
    od, on_, oc = d.clone(), n.clone(), c.clone()
    y, x, qy, qx = ys[ok], xs[ok], by[ok], bx[ok]
    od[y, x], on_[y, x], oc[y, x] = dn[ok], n[qy, qx], c[qy, qx]
    return _np(od), _np(on_), _np(oc), None, None


def _exact_fuse(case, seed):
    sc, src = _terrain(case, seed)
    maps = _maps(sc, seed)
    p = fusion.FusionParams()
    cos_n, r2 = math.cos(math.radians(p.max_normal_error_deg)), p.max_reproj_error ** 2
    dep, nrm, cst = ([_t(m[i]) for m in maps] for i in range(3))
    used = [torch.zeros_like(d, dtype=torch.bool) for d in dep]
    cams = [(v.k, _t(np.asarray(v.r, float)), _t(np.asarray(v.t, float))) for v in sc.views]
    base = [_median_distance(sc, v, src[v]) for v in range(len(maps))]
    h, w = dep[0].shape

    def lift(cam, x, y, d):
        k, r, t = cam
        return (torch.stack([(x - k[2]) / k[0] * d, (y - k[3]) / k[1] * d, d], -1) - t) @ r

    def project(cam, x):
        k, r, t = cam
        q = x @ r.T + t
        return k[0] * q[:, 0] / q[:, 2] + k[2], k[1] * q[:, 1] / q[:, 2] + k[3], q[:, 2]

    def weight(v, y, x, d):
        s = d * d * (p.sigma_px0 + p.sigma_px_slope * cst[v][y, x].clamp(0, 2)) / (cams[v][0][0] * base[v])
        return 1 / (s * s).clamp(min=1e-300)

    pos, nor = [], []
    for v in range(len(maps)):
        y, x = torch.nonzero((dep[v] > 0) & ~used[v], as_tuple=True)
        d = dep[v][y, x]
        xw = lift(cams[v], x.to(F), y.to(F), d)
        nw = nrm[v][y, x] @ cams[v][1]
        g = weight(v, y, x, d)[:, None]
        sw, sx, sn = g, g * xw, g * nw
        hits = []
        for o in src[v][: p.consistency_num_images]:
            u, q, z = project(cams[o], xw)
            cu, rv = torch.floor(u + 0.5), torch.floor(q + 0.5)
            ok = (z > 0) & (cu >= 0) & (rv >= 0) & (cu < w) & (rv < h)
            yo, xo = torch.nan_to_num(rv).clamp(0, h - 1).long(), torch.nan_to_num(cu).clamp(0, w - 1).long()
            od = dep[o][yo, xo]
            ok &= (od > 0) & ~((z - od).abs() / od > p.max_depth_error)
            xx = lift(cams[o], xo.to(F), yo.to(F), od)
            bu, bv, bz = project(cams[v], xx)
            ok &= (bz > 0) & ~((bu - x) ** 2 + (bv - y) ** 2 > r2)
            no = nrm[o][yo, xo] @ cams[o][1]
            ok &= ~((no * nw).sum(-1) < cos_n)
            g = torch.where(ok, weight(o, yo, xo, od), 0.0)[:, None]
            sw, sx, sn = sw + g, sx + g * torch.nan_to_num(xx), sn + g * no
            hits.append((o, ok, yo, xo))
        length = sn.norm(dim=-1)
        take = (sum(hit[1].long() for hit in hits) >= p.min_consistent_views) & (length >= 2.0 ** -23)
        for o, ok, yo, xo in hits:
            used[o][yo[ok & take], xo[ok & take]] = True
        pos.append((sx / sw)[take])
        nor.append((sn / length[:, None])[take])
    whole = np.zeros((2, sum(m[0].size for m in maps), 3))
    for a, b in zip(whole, (pos, nor)):
        b = _np(torch.cat(b))
        a[: len(b)] = b
    return whole[0], whole[1], None, None, None


def _median_distance(sc, v, sources):
    c = sc.views[v].center()
    return float(np.quantile([np.linalg.norm(c - sc.views[s].center()) for s in sources], 0.5))


def _exact_scene(case, seed):
    sc = _tracks(case, seed)
    ctr = np.array([v.center() for v in sc.views])
    n = len(sc.views)
    pair, ang = [], []
    by_view = [[] for _ in range(n)]
    for p in sc.points:
        vs = np.array(p.views)
        for v in vs:
            z = float(sc.views[v].r[2] @ p.xyz + sc.views[v].t[2])
            if z > 0:
                by_view[v].append(z)
        e = ctr[vs] - p.xyz
        e /= np.linalg.norm(e, axis=1, keepdims=True)
        i, j = np.tril_indices(len(vs), -1)
        a = np.arccos(np.clip((e[i] * e[j]).sum(1), -1, 1))
        pair.append(np.minimum(vs[i], vs[j]) * n + np.maximum(vs[i], vs[j]))
        ang.append(np.minimum(a, math.pi - a))
    pair, ang = np.concatenate(pair), np.concatenate(ang)
    order = np.lexsort((ang, pair))
    pair, ang = pair[order], ang[order]
    q75 = np.zeros((n, n))
    ids, start, cnt = np.unique(pair, return_index=True, return_counts=True)
    for g, s, c in zip(ids, start, cnt):
        q75[g // n, g % n] = q75[g % n, g // n] = np.quantile(ang[s : s + c], 0.75)
    ranges = np.zeros((n, 2))
    for v, z in enumerate(by_view):
        if z:
            z = sorted(z)
            ranges[v] = 0.75 * z[min(int(len(z) * 0.01), len(z) - 1)], 1.25 * z[min(int(len(z) * 0.99), len(z) - 1)]
    return None, q75, None, ranges


# (input channels, output channels, kernel side, halvings of the resolution) of each layer in order
_LAYERS = [(64, 32, 3, 0), (32, 32, 3, 0), (32, 64, 3, 1), (64, 64, 3, 1), (64, 128, 3, 2), (128, 128, 3, 2), (128, 128, 3, 3),
           (128, 128, 3, 3), (256, 128, 3, 2), (192, 64, 3, 1), (96, 32, 3, 0), (32, 32, 1, 0)]


def _sweep_features(views, case):
    """The network's 64 input channels: 32 sweep costs, the intensity, zeros; in the bf16 that the
    network takes."""
    hh, ww = _net_size(case)
    out = []
    for gray, k, sources in views:
        ref = _t(gray)
        h, w = ref.shape
        ray, _, _ = _rays(np.asarray(k, np.float32).astype(np.float64), h, w, ref.device)
        f = torch.zeros(hh, ww, 64, dtype=F, device=ref.device)
        for q in range(32):
            d = 1 / (1 / FAR + (q + 0.5) / 32 * (1 / NEAR - 1 / FAR))
            cost, cnt = torch.zeros_like(ref), torch.zeros_like(ref)
            for g, ks, r, t in sources:
                p = (ray * d) @ _t(np.asarray(r).reshape(3, 3)).T + _t(np.asarray(t))
                u, v = ks[0] * p[..., 0] / p[..., 2] + ks[2], ks[1] * p[..., 1] / p[..., 2] + ks[3]
                ok = (p[..., 2] > 1e-6) & (u >= 0) & (v >= 0) & (u <= g.shape[1] - 1) & (v <= g.shape[0] - 1)
                cost += torch.where(ok, (ref - _bilinear(_t(g), u, v)).abs(), 0.0)
                cnt += ok
            f[:h, :w, q] = torch.where(cnt > 0, cost / (255 * cnt.clamp(min=1)), 1.0)
        f[:h, :w, 32] = ref / 255
        out.append(f.to(torch.float32).to(torch.bfloat16).to(F))
    return torch.stack(out)


def _unet(params, x):
    """The U-Net on (batch, h, w, channels) from the flat parameter vector."""
    at = 0

    def layer(i, x, relu=True):
        nonlocal at
        cin, cout, k, _ = _LAYERS[i]
        wgt = params[at : at + cout * k * k * cin].reshape(cout, k, k, cin)
        bias = params[at + cout * k * k * cin : at + cout * k * k * cin + cout]
        at += cout * k * k * cin + cout
        b, h, w, _ = x.shape
        r = k // 2
        xp = torch.nn.functional.pad(x, (0, 0, r, r, r, r))
        y = bias
        for a in range(k):
            for c in range(k):
                y = y + (xp[:, a : a + h, c : c + w].reshape(-1, cin) @ wgt[:, a, c].T).reshape(b, h, w, cout)
        return torch.relu(y) if relu else y

    def pool(x):
        return (x[:, ::2, ::2] + x[:, 1::2, ::2] + x[:, ::2, 1::2] + x[:, 1::2, 1::2]) / 4

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    e0 = layer(1, layer(0, x))
    e1 = layer(3, layer(2, pool(e0)))
    e2 = layer(5, layer(4, pool(e1)))
    e3 = layer(7, layer(6, pool(e2)))
    d2 = layer(8, torch.cat([up(e3), e2], -1))
    d1 = layer(9, torch.cat([up(d2), e1], -1))
    d0 = layer(10, torch.cat([up(d1), e0], -1))
    return layer(11, d0, relu=False)


def _exact_predict(case, seed):
    _, views = _sweep_views(case, seed)
    with torch.no_grad():
        o = _unet(_t(_weights()), _sweep_features(views, case))[..., :5]
    depth = 1 / (1 / FAR + torch.sigmoid(o[..., 0]) * (1 / NEAR - 1 / FAR))
    normal = o[..., 1:4] / torch.sqrt((o[..., 1:4] ** 2).sum(-1, keepdim=True) + 1e-6)
    return _np(depth), _np(normal), _np(torch.sigmoid(o[..., 4])), _np(o)


def _exact_train(case, seed):
    sc, views = _sweep_views(case, seed)
    labels = [_labels(sc, case, b) for b in range(case["batch"])]
    d, n = _t(np.stack([q[0] for q in labels])), _t(np.stack([q[1] for q in labels]))
    p = _t(_weights()).requires_grad_()
    t = init_net.TrainParams()
    o = _unet(p, _sweep_features(views, case))
    on = d > 0
    inv = 1 / FAR + torch.sigmoid(o[..., 0]) * (1 / NEAR - 1 / FAR)
    ld = ((inv - 1 / torch.where(on, d, 1.0)).abs() / (1 / NEAR - 1 / FAR))[on].sum()
    nv = o[..., 1:4] / torch.sqrt((o[..., 1:4] ** 2).sum(-1, keepdim=True) + 1e-6)
    ln = (1 - (nv * n).sum(-1))[on].sum()
    close = ((1 / inv - d).abs() <= t.conf_tol * d).to(F).detach()
    lc = torch.nn.functional.binary_cross_entropy_with_logits(o[..., 4], close, reduction="none")[on].sum()
    (ld + t.w_normal * ln + t.w_conf * lc).backward()
    return np.array([float(ld), float(ln), float(lc), float(on.sum())]), _np(p.grad)


def exact(case, seed):
    """`run`'s outputs in 64 bits; None for a PatchMatch search, whose random walk has no such value."""
    how = {"readout": _exact_readout, "post": _exact_post, "fuse": _exact_fuse, "scene": _exact_scene, "predict": _exact_predict,
           "train": _exact_train}.get(case["kind"])
    return how(case, seed) if how else None
