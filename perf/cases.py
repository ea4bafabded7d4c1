"""The work that a user of this renderer has it do, as measurable cases.

A case is a dict of plain values; ``kind`` says which entry point it goes
through:

  frame        HipRenderer.render_frame: one progressive sample, the
               contract call of the interactive preview (latency and
               launches count)
  render       HipRenderer.render: a still of ``spp`` samples per pixel from
               a cleared accumulation, image returned to the host
  guided       the same with a trained-and-frozen guiding network (final
               frames after training)
  jobs         HipRenderer.render_jobs: a list of uneven jobs over several
               resident scenes, one call
  trace        HipRenderer.trace_closest and trace_any on host ray batches
               (picking, baking, parity checks)
  blas_build   HipRenderer.build_blas: acceleration structure of a new mesh
  blas_refit   HipRenderer.refit_blas: the boxes of a deforming mesh
  output       image_rgb8 and noise_stats of a host framebuffer (what
               save_image computes before it writes the file)
  guide_train  HipRenderer.guide_train on a host batch, gradients returned
  guide_sample HipRenderer.guide_sample: directions and pdfs at host points

Scenes and sizes are those of xenon_amd.scenes' generators, the tests and
bench.py; inputs (camera position, first sample index, rays, vertices,
framebuffers, network parameters) are made from the seed.
"""
import dataclasses
import math

import numpy as np

from xenon_amd import HipRenderer, HipScene, GpuScene, scenes

F32 = np.float32
LEVELS, FEATURES = 16, 2
LAYERS = ((48, 64), (64, 64), (64, 64), (64, 48))

# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # interactive preview of a small frame: the smallest render call
        dict(name="frame_cornell_256", kind="frame", scene="cornell", width=256, height=256, depth=8),
        # interactive preview at full resolution on the large mesh
        dict(name="frame_mesh_1080p", kind="frame", scene="mesh8", width=1920, height=1080, depth=8),
        # the box rendered to 64 samples: closed scene, long paths, area light
        dict(name="cornell_512_64spp", kind="render", scene="cornell", width=512, height=512, spp=64, depth=8),
        # the headline workload: 1.3M-triangle mesh, sun and sky
        dict(name="mesh_1080p_256spp", kind="render", scene="mesh8", width=1920, height=1080, spp=256, depth=8),
        # 4096 instances of ten meshes, mixed materials, depth 10
        dict(name="instancing_1080p_64spp", kind="render", scene="inst4096", width=1920, height=1080, spp=64,
             depth=10),
        # analytic primitives beside meshes, every lobe, an odd resolution and sample count
        dict(name="prims_801x449_33spp", kind="render", scene="prims", width=801, height=449, spp=33, depth=8),
        # final frame of the caustic room with a frozen guide, one full guided batch
        dict(name="guided_room_720p_72spp", kind="guided", scene="room", width=1280, height=720, spp=72, depth=8,
             t_log2=19),
        # a queue of eight uneven jobs in one call
        dict(name="jobs_8_mixed", kind="jobs", jobs=8, list_seed=6, lo=256, hi=768, spp_max=64),
        # a million host rays, closest hit and any hit
        dict(name="trace_mesh_1m", kind="trace", scene="mesh8", rays=1 << 20),
        # a new 300k-triangle mesh
        dict(name="blas_build_300k", kind="blas_build", tris=300000),
        # saving a 1080p image: 8-bit conversion and noise statistics
        dict(name="output_1080p", kind="output", width=1920, height=1080),
        # one training step of the guide on a host batch
        dict(name="guide_train_64k", kind="guide_train", points=1 << 16, t_log2=15),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "render", "render", "render", "guided", "jobs", "trace", "trace", "blas_build",
                       "blas_refit", "output", "guide_train", "guide_sample"])
    if kind in ("frame", "render"):
        scene = rng.choice(["cornell", "mesh4", "mesh6", "mesh8", "inst512", "prims", "room"])
        w, h = _log(rng, 64, 1920), _log(rng, 64, 1080)
        c = dict(kind=kind, scene=scene, width=w, height=h, depth=rng.randint(4, 12))
        if kind == "render":
            most = (1 << 26) if scene in ("inst512", "prims") else (1 << 27)
            c["spp"] = _log(rng, 1, max(1, min(256, most // (w * h))))
        return c
    if kind == "guided":
        w, h = _log(rng, 160, 1280), _log(rng, 90, 720)
        return dict(kind=kind, scene="room", width=w, height=h, spp=_log(rng, 4, 72), depth=rng.randint(6, 10),
                    t_log2=rng.randint(15, 19))
    if kind == "jobs":
        lo = rng.randrange(128, 400, 16)
        return dict(kind=kind, jobs=rng.randint(2, 12), list_seed=rng.randint(0, 9999), lo=lo,
                    hi=lo + 16 * rng.randint(4, 24), spp_max=rng.choice([16, 32, 64]))
    if kind == "trace":
        return dict(kind=kind, scene=rng.choice(["cornell", "mesh6", "mesh8", "inst512", "prims"]),
                    rays=_log(rng, 64, 1 << 20))
    if kind in ("blas_build", "blas_refit"):
        return dict(kind=kind, tris=_log(rng, 500, 1300000))
    if kind == "output":
        return dict(kind=kind, width=_log(rng, 64, 3840), height=_log(rng, 64, 2160))
    return dict(kind=kind, points=_log(rng, 500, 1 << 18), t_log2=rng.randint(14, 17))


# ---------------------------------------------------------------------------
# what a program has in hand
# ---------------------------------------------------------------------------

_scenes = {}     # built host scenes by name: a program builds (or loads) its scene once
_meshes = {}


def _desc(name):
    if name == "cornell":
        return scenes.cornell()
    if name.startswith("mesh"):
        return scenes.big_mesh(level=int(name[4:]))
    if name == "inst4096":
        return scenes.instancing()
    if name == "inst512":
        return scenes.instancing(n_inst=512, tri_range=(2000, 20000), n_emit=16)
    if name == "prims":
        return scenes.prim_shapes()
    return scenes.caustic_room()


def _scene(name):
    if name not in _scenes:
        _scenes[name] = HipScene(_desc(name))
    return _scenes[name]


def _camera(scene, rng, width, height):
    """The scene's camera moved a little, as a program that walks through it does."""
    home = scene.desc.camera
    far = np.linalg.norm(np.subtract(home.eye, home.target))
    move = rng.uniform(-0.01, 0.01, 3) * far
    scene.desc.camera = dataclasses.replace(home, eye=tuple(float(x) for x in np.add(home.eye, move)))
    try:
        return scene.camera(width, height)
    finally:
        scene.desc.camera = home


def _unit(rng, n):
    v = rng.standard_normal((n, 3)).astype(F32)
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def _bounds(scene):
    lo, hi = scene.bounds()
    return np.clip(lo, -50, 150).astype(F32), np.clip(hi, -50, 150).astype(F32)


def _rays(scene, n, rng):
    """Half camera rays, half rays between random points of the scene's box: (closest-hit rays, any-hit segments)."""
    lo, hi = _bounds(scene)
    cam = _camera(scene, rng, 1920, 1080)
    eye, llc, hz, vt = (np.array(v[:], F32) for v in (cam.eye, cam.lower_left, cam.horizontal, cam.vertical))
    k = n // 2
    st = rng.random((k, 2)).astype(F32)
    d = llc + st[:, :1] * hz + st[:, 1:] * vt - eye
    a = np.concatenate([np.broadcast_to(eye, (k, 3)), d], 1)
    p, q = (lo + rng.random((n - k, 3)).astype(F32) * (hi - lo) for _ in range(2))
    od = np.concatenate([a, np.concatenate([p, q - p], 1)])
    length = np.linalg.norm(od[:, 3:], axis=1, keepdims=True).astype(F32)
    od[:, 3:] /= length
    close = np.concatenate([od, np.full((n, 1), 1e-4, F32), np.full((n, 1), np.inf, F32)], 1)
    seg = close.copy()
    seg[:, 6] = 5e-4
    seg[:, 7] = length[:, 0]
    return np.ascontiguousarray(close, F32), np.ascontiguousarray(seg, F32)


def _mesh(tris, seed):
    """`tris` triangles of a subdivided sphere, displaced by a smooth function of the seed."""
    level = 0
    while 20 * 4 ** level < tris:
        level += 1
    if level not in _meshes:
        _meshes[level] = scenes.icosphere(level)
    V, T = _meshes[level]
    rng = np.random.default_rng(seed)
    r = np.ones(V.shape[0])
    for _ in range(3):
        r += 0.03 * np.sin(V @ rng.uniform(-9, 9, 3) + rng.uniform(0, 6.3))
    return (V * r[:, None]).astype(F32), np.ascontiguousarray(T[:tris], np.int32)


def _network(seed, t_log2):
    rng = np.random.default_rng(seed + 77)
    grid = (rng.random((LEVELS, 1 << t_log2, FEATURES), dtype=F32) - F32(0.5)) * F32(0.4)
    w = [rng.uniform(-1, 1, d).astype(F32) * F32(math.sqrt(6.0 / sum(d))) for d in LAYERS]
    return grid, np.concatenate([x.ravel() for x in w])


def _image(case, seed):
    """A smooth picture with the noise of a few samples per pixel."""
    rng = np.random.default_rng(seed)
    h, w = case["height"], case["width"]
    y, x = np.mgrid[0:h, 0:w].astype(F32)
    base = 0.4 + 0.3 * np.sin(x / 97 + rng.uniform(0, 6)) * np.cos(y / 61 + rng.uniform(0, 6))
    return (np.exp(0.2 * rng.standard_normal((h, w, 3), dtype=F32)) * base[..., None].astype(F32)).astype(F32)


def _points(n, seed):
    rng = np.random.default_rng(seed)
    return dict(pos=rng.random((n, 3)).astype(F32), nrm=_unit(rng, n), dirs=_unit(rng, n),
                lam=np.exp(rng.standard_normal(n)).astype(F32), u=rng.random((n, 3)).astype(F32))


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = dict(case)
    if kind in ("frame", "render", "guided"):
        scene = _scene(case["scene"])
        w, h = case["width"], case["height"]
        # a guided batch holds at most 2^26 paths: the guided program sizes its queues for one
        lim = case["spp"] if kind == "guided" else 0
        r = s["renderer"] = HipRenderer(w, h, case["depth"], scene.desc.min_bounces, spp_per_launch=lim)
        r.upload_scene(scene)
        s["camera"] = _camera(scene, rng, w, h)
        s["first"] = int(rng.integers(1, 1 << 20))
        if kind == "guided":
            r.guide_enable(t_log2=case["t_log2"], seed=seed & 0xFFFF)
            r.guide_set_params(*_network(seed, case["t_log2"]))
            r.guide_set_training(False)
    elif kind == "jobs":
        # a farm's context: queues of 2^26 paths, more than most of its jobs need
        r = s["renderer"] = HipRenderer(1024, 1024, 8, 3, spp_per_launch=64)
        todo = scenes.job_list(case["jobs"], case["list_seed"], (case["lo"], case["hi"]),
                               tuple(x for x in (16, 32, 64) if x <= case["spp_max"]))
        gpu, s["work"] = {}, []
        for j in todo:
            if j.kind not in gpu:
                scene = _scene(("cornell", "mesh6", "inst512")[j.kind])
                gpu[j.kind] = GpuScene(r, scene)
            scene = gpu[j.kind].scene
            s["work"].append(dict(scene=gpu[j.kind], camera=_camera(scene, rng, j.width, j.height), width=j.width,
                                  height=j.height, spp_first=int(rng.integers(1, 1 << 20)), spp_count=j.spp,
                                  max_bounces=j.max_bounces, min_bounces=3))
    elif kind == "trace":
        scene = _scene(case["scene"])
        r = s["renderer"] = HipRenderer(64, 64)
        r.upload_scene(scene)
        s["close"], s["segments"] = _rays(scene, case["rays"], rng)
    elif kind in ("blas_build", "blas_refit"):
        r = s["renderer"] = HipRenderer(64, 64)
        s["pos"], s["idx"] = _mesh(case["tris"], seed)
        if kind == "blas_refit":
            s["nodes"], s["prims"] = r.build_blas(*_mesh(case["tris"], 0))
    elif kind == "output":
        s["renderer"] = HipRenderer(64, 64)
        s["rgb"] = _image(case, seed)
    else:
        r = s["renderer"] = HipRenderer(8, 8, 4, 2)
        r.guide_enable((0, 0, 0), (1, 1, 1), t_log2=case["t_log2"], seed=seed & 0xFFFF)
        r.guide_set_params(*_network(seed, case["t_log2"]))
        s.update(_points(case["points"], seed))
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(s):
    r, kind = s["renderer"], s["kind"]
    if kind == "frame":
        return r.render_frame(s["camera"])
    if kind in ("render", "guided"):
        r.reset()
        return r.render(s["camera"], s["first"], s["spp"])
    if kind == "jobs":
        return r.render_jobs(s["work"])
    if kind == "trace":
        hits = r.trace_closest(s["close"])
        return {"occluded": r.trace_any(s["segments"]), **{k: hits[k] for k in hits.dtype.names}}
    if kind == "blas_build":
        nodes, prims = r.build_blas(s["pos"], s["idx"])
        return {"prims": prims, **{k: nodes[k] for k in nodes.dtype.names}}
    if kind == "blas_refit":
        nodes = r.refit_blas(s["pos"], s["idx"], s["nodes"], s["prims"])
        return {k: nodes[k] for k in nodes.dtype.names}
    if kind == "output":
        return {"rgb8": r.image_rgb8(s["rgb"]), "stats": r.noise_stats(s["rgb"])}
    if kind == "guide_train":
        loss, grid, w = r.guide_train(s["pos"], s["nrm"], s["dirs"], s["lam"], apply=False, want_grads=True)
        return {"loss": loss, "grid": grid, "weights": w}
    d, pdf = r.guide_sample(s["pos"], s["nrm"], s["u"])
    return {"dir": d, "pdf": pdf}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

# per scene: rays per path (closest + shadow) in earnest, triangles
_SHAPE = {"cornell": (5.8, 36), "mesh4": (2.7, 5122), "mesh6": (2.7, 81922), "mesh8": (2.7, 1310722),
          "inst512": (2.1, 100000), "inst4096": (2.1, 700000), "prims": (3.0, 400), "room": (5.0, 499310)}


def _ray_flops(tris):
    """A box pair per level of the tree (26 operations a box), a triangle test."""
    return 52.0 * max(1.0, math.log2(tris)) + 50.0


def _path_work(scene, paths, pixels):
    rays, tris = _SHAPE[scene]
    return {"bytes": 112.0 * tris + 12.0 * pixels, "flops": paths * (rays * _ray_flops(tris) + 300.0)}


def work(case):
    kind = case["kind"]
    if kind in ("frame", "render", "guided"):
        px = case["width"] * case["height"]
        w = _path_work(case["scene"], px * case.get("spp", 1), px)
        if kind == "guided":   # one network query per pixel: 32 x 8 corners, four layers
            w["bytes"] += px * 512.0
            w["flops"] += px * 2.0 * sum(a * b for a, b in LAYERS)
        return w
    if kind == "jobs":
        total = {"bytes": 0.0, "flops": 0.0}
        for j in scenes.job_list(case["jobs"], case["list_seed"], (case["lo"], case["hi"]),
                                 tuple(x for x in (16, 32, 64) if x <= case["spp_max"])):
            px = j.width * j.height
            w = _path_work(("cornell", "mesh6", "inst512")[j.kind], px * j.spp, px)
            total = {k: total[k] + w[k] for k in total}
        return total
    if kind == "trace":
        _, tris = _SHAPE[case["scene"]]
        n = case["rays"]
        return {"bytes": n * (2 * 32.0 + 64.0 + 1.0) + 80.0 * tris, "flops": 2.0 * n * _ray_flops(tris)}
    if kind in ("blas_build", "blas_refit"):
        n = case["tris"]   # vertices and indices in, nodes and leaf slots out
        return {"bytes": 6.0 * n + 12.0 * n + 64.0 * n + 4.0 * n * (2 if kind == "blas_refit" else 1),
                "flops": 40.0 * n}
    if kind == "output":
        px = case["width"] * case["height"]
        return {"bytes": px * (2 * 12.0 + 3.0), "flops": px * 60.0}
    n, t = case["points"], 1 << case["t_log2"]
    macs = sum(a * b for a, b in LAYERS)
    if kind == "guide_train":
        return {"bytes": n * 40.0 + n * 1024.0 + LEVELS * t * 8.0 + macs * 8.0, "flops": 6.0 * n * macs}
    return {"bytes": n * 52.0 + n * 512.0, "flops": 2.0 * n * macs}


# ---------------------------------------------------------------------------
# values in 64 bits
# ---------------------------------------------------------------------------


def _exact_output(rgb):
    """Residual noise statistics (luminance, 1-2-1 blur, edge mask, normalised residuals)."""
    a = rgb.astype(np.float64)
    h, w = a.shape[:2]
    lum = 0.2126 * a[..., 0] + 0.7152 * a[..., 1] + 0.0722 * a[..., 2]
    names = ("mean_squared_score", "rms_score", "mean_absolute", "median_absolute", "p95_absolute", "max_absolute",
             "avg_luminance", "edge_threshold", "epsilon")
    avg = lum.mean()
    edge, eps = max(1e-6, avg * 0.1), max(1e-8, avg * avg * 1e-4)
    c = lum[1:-1, 1:-1]
    gx, gy = 0.5 * (lum[1:-1, 2:] - lum[1:-1, :-2]), 0.5 * (lum[2:, 1:-1] - lum[:-2, 1:-1])
    keep = np.hypot(gx, gy) < edge
    k = np.array([1.0, 2.0, 1.0])
    blur = sum(k[i] * k[j] * lum[i:h - 2 + i, j:w - 2 + j] for i in range(3) for j in range(3)) / 16.0
    res, den = (c - blur)[keep], (blur * blur + eps)[keep]
    q2, q1 = res * res / den, np.sort(np.abs(res) / np.sqrt(den))
    n = q1.size
    got = dict.fromkeys(names, 0.0)
    got.update(avg_luminance=avg, edge_threshold=edge, epsilon=eps)
    if n:
        got.update(mean_squared_score=q2.mean(), rms_score=math.sqrt(q2.mean()), mean_absolute=q1.mean(),
                   median_absolute=q1[int(F32(0.5) * F32(n - 1))], p95_absolute=q1[int(F32(0.95) * F32(n - 1))],
                   max_absolute=q1[-1])
    return {"rgb8": None, "stats": {**{m: float(v) for m, v in got.items()}, "valid_pixel_count": int(n),
                                    "total_interior_pixel_count": (w - 2) * (h - 2),
                                    "valid_pixel_ratio": n / ((w - 2) * (h - 2))}}


def _encode(torch, p, nrm, grid, t_log2):
    """Hash-grid features (16 levels, trilinear) and the 16 real spherical harmonics of the normal, in 64 bits."""
    T = 1 << t_log2
    b = math.exp((math.log(2048.0) - math.log(16.0)) / (LEVELS - 1))
    cols = []
    for lv in range(LEVELS):
        res = int(math.floor(16.0 * b ** lv))
        # the lattice cell and the weights are of the position as given, in 32 bits
        x = np.clip(p, F32(0), F32(0.99999994)) * F32(res)
        i0 = np.floor(x).astype(np.int64)
        f = torch.from_numpy((x - i0.astype(F32)).astype(np.float64))
        acc = 0.0
        for c in range(8):
            o = np.array([c & 1, c >> 1 & 1, c >> 2 & 1])
            ix = i0 + o
            n = res + 1
            if n ** 3 <= T:
                at = ix[:, 0] + ix[:, 1] * n + ix[:, 2] * n * n
            else:
                hsh = ix.astype(np.uint64) * np.array([1, 2654435761, 805459861], np.uint64)
                at = ((hsh[:, 0] ^ hsh[:, 1] ^ hsh[:, 2]) & np.uint64(T - 1)).astype(np.int64)
            wt = torch.ones(len(p), dtype=torch.float64)
            for a in range(3):
                wt = wt * (f[:, a] if o[a] else 1 - f[:, a])
            acc = acc + wt[:, None] * grid[lv][torch.from_numpy(at)]
        cols.append(acc)
    x, y, z = (torch.from_numpy(nrm.astype(np.float64))[:, k] for k in range(3))
    s = [0.28209479177387814 + 0 * x, -0.48860251190291987 * y, 0.48860251190291987 * z, -0.48860251190291987 * x,
         1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.94617469575755997 * z * z - 0.31539156525251999,
         -1.0925484305920792 * x * z, 0.54627421529603959 * (x * x - y * y),
         0.59004358992664352 * y * (-3 * x * x + y * y), 2.8906114426405538 * x * y * z,
         0.45704579946446572 * y * (1 - 5 * z * z), 0.3731763325901154 * z * (5 * z * z - 3),
         0.45704579946446572 * x * (1 - 5 * z * z), 1.4453057213202769 * z * (x * x - y * y),
         0.59004358992664352 * x * (-x * x + 3 * y * y)]
    return torch.cat([*cols, torch.stack(s, 1)], 1)


def _mixture(torch, out):
    raw = out[:, :40].reshape(-1, 8, 5)
    m = raw[..., :3]
    mu = m / torch.sqrt((m * m).sum(-1, keepdim=True) + 1e-12)
    return mu, torch.exp(raw[..., 3].clamp(-4.0, 8.0)), torch.softmax(raw[..., 4], -1)


def _pdf(torch, mu, kappa, pi, w):
    lobes = kappa / (2 * math.pi * -torch.expm1(-2 * kappa)) * torch.exp(kappa * ((mu * w[:, None]).sum(-1) - 1))
    return (pi * lobes).sum(-1)


def _exact_guide(case, seed):
    import torch
    grid, w = _network(seed, case["t_log2"])
    pts = _points(case["points"], seed)
    n = case["points"]
    train = case["kind"] == "guide_train"
    G = torch.from_numpy(grid.astype(np.float64)).requires_grad_(train)
    W, at = [], 0
    for a, b in LAYERS:
        W.append(torch.from_numpy(w[at:at + a * b].reshape(a, b).astype(np.float64)).requires_grad_(train))
        at += a * b
    h = _encode(torch, pts["pos"], pts["nrm"], G, case["t_log2"])
    for k, m in enumerate(W):
        h = h @ m
        h = torch.relu(h) if k < 3 else h
    if train:
        lam = torch.from_numpy(pts["lam"].astype(np.float64))
        lam = lam * (n / lam.sum())
        leaf = h.detach().requires_grad_(True)
        q = _pdf(torch, *_mixture(torch, leaf), torch.from_numpy(pts["dirs"].astype(np.float64)))
        loss = -lam * torch.log(q.clamp_min(1e-20))
        (g,) = torch.autograd.grad(loss.sum(), leaf)
        h.backward(g.clamp(-1024.0, 1024.0))
        return {"loss": float(loss.detach().mean()), "grid": G.grad.numpy(),
                "weights": np.concatenate([m.grad.numpy().ravel() for m in W])}
    mu, kappa, pi = _mixture(torch, h)
    u = torch.from_numpy(pts["u"].astype(np.float64))
    j = (torch.cumsum(pi, 1) < u[:, :1]).sum(1).clamp_max(7)
    row = torch.arange(n)
    m, k = mu[row, j], kappa[row, j]
    wz = 1 + torch.log(u[:, 1] + (1 - u[:, 1]) * torch.exp(-2 * k)) / k
    st = torch.sqrt((1 - wz * wz).clamp_min(0))
    phi = 2 * math.pi * u[:, 2]
    sg = torch.where(m[:, 2] >= 0, 1.0, -1.0).double()
    a = -1 / (sg + m[:, 2])
    b = m[:, 0] * m[:, 1] * a
    t1 = torch.stack([1 + sg * m[:, 0] ** 2 * a, sg * b, -sg * m[:, 0]], 1)
    t2 = torch.stack([b, sg + m[:, 1] ** 2 * a, -m[:, 1]], 1)
    d = (st * torch.cos(phi))[:, None] * t1 + (st * torch.sin(phi))[:, None] * t2 + wz[:, None] * m
    return {"dir": d.numpy(), "pdf": _pdf(torch, mu, kappa, pi, d).numpy()}


def _exact_hits(rays, desc):
    """Every triangle of a one-mesh scene against every ray: the nearest hit's distance and barycentrics."""
    P = desc.meshes[0].positions.astype(np.float64)
    T = desc.meshes[0].indices
    best = np.full(len(rays), np.inf)
    uv = np.zeros((len(rays), 2))
    o, d = rays[:, :3].astype(np.float64), rays[:, 3:6].astype(np.float64)
    tmin = rays[:, 6].astype(np.float64)
    for i0, i1, i2 in T:
        e1, e2 = P[i1] - P[i0], P[i2] - P[i0]
        hh = np.cross(d, e2)
        det = hh @ e1
        ok = np.abs(det) >= 1e-7
        inv = 1.0 / np.where(ok, det, 1.0)
        s = o - P[i0]
        u = inv * (s * hh).sum(1)
        q = np.cross(s, e1)
        v = inv * (d * q).sum(1)
        t = inv * (q @ e2)
        ok &= (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= tmin) & (t <= best)
        best[ok] = t[ok]
        uv[ok, 0], uv[ok, 1] = u[ok], v[ok]
    return best, uv


def exact(case, seed):
    kind = case["kind"]
    if kind in ("guide_train", "guide_sample"):
        return _exact_guide(case, seed)
    if kind == "output":
        return _exact_output(_image(case, seed))
    if kind == "trace" and case["scene"] == "cornell":
        rays, _ = _rays(_scene("cornell"), case["rays"], np.random.default_rng(seed))
        t, uv = _exact_hits(rays, _desc("cornell"))
        none = dict.fromkeys(("occluded", "instance_id", "prim_id", "mat_id", "pos", "normal", "geo_normal",
                              "front_face"))
        return {"t": t, "u": uv[:, 0], "v": uv[:, 1], **none}
    # a path-traced image has no value in 64 bits that could be had in time: every sample's path depends on the
    # 32-bit roundings of the hits before it
    return None
