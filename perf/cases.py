"""Workloads of the renderer, from the smallest call to the largest, each one
pass through the public Python entry points.

A case is a dict of plain values; `kind` names the entry point:

  nee      wr.render_nee: NEE + MIS path tracing of one frame (vacuum, medium,
           or with an envmap light)
  light    wr.render_light: light subpaths splatted to the camera
  bdpt     wr.render_bdpt: bidirectional path tracing
  guided   wr.render_guided with a network the caller holds (no training
           between passes: a training render's records arrive in an order of
           their own, so its images are a different sample every time)
  train    Guide.train: Adam steps on records the caller has (steps > 0), or
           Guide.gradient (steps = 0)
  batch    wr.render_batch: many small jobs in one path pool
  first    a scene from its host mesh (BVH build, tables) and its first frame
  trace    GpuScene.trace_closest / trace_any of rays the caller has

Renders return the FP32 image a program writes out (scenes.write_pfm).  The
scenes are the generators of wurstrenderer_amd/scenes.py; sizes follow bench.py
and the tests: 64^2 previews to the 1920 x 1080, 64-spp frame over 1.31 million
triangles.
"""
from __future__ import annotations

import math

import numpy as np

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

SKY = 256  # texel rows of the envmap of cases with env=True

# The largest frame: 1920 x 1080 at 64 spp and 18 path vertices.  Drawn cases
# stay below these counts of samples and of samples x path vertices.
MOST_SAMPLES = 1920 * 1080 * 64


def listed():
    return [
        # an interactive preview: the smallest frame, bound by launches and polls
        dict(name="preview_64", kind="nee", scene="cornell", tris=36, width=64, height=64, spp=4, vertices=10,
             medium=False, env=False),
        # the Cornell workload of the tests
        dict(name="cornell_256", kind="nee", scene="cornell", tris=36, width=256, height=256, spp=64, vertices=10,
             medium=False, env=False),
        # the headline frame of bench.py
        dict(name="spheres_1080p", kind="nee", scene="spheres", tris=1310720, width=1920, height=1080, spp=64,
             vertices=18, medium=False, env=False),
        # an interior lit through a gap: nearly all shadow rays are occluded; an odd resolution
        dict(name="room_odd", kind="nee", scene="room", tris=1003520, width=961, height=541, spp=24, vertices=18,
             medium=False, env=False),
        # a foggy interior: free flights, phase function, deep paths
        dict(name="fog_360p", kind="nee", scene="clutter", tris=716800, width=640, height=360, spp=32, vertices=34,
             medium=True, env=False),
        # path guiding with a trained network: inference at every vertex
        dict(name="guided_540p", kind="guided", scene="room", tris=1003520, width=960, height=540, spp=16, vertices=18,
             fp8=False),
        # training the guiding network on a quarter of a million records
        dict(name="train_256k", kind="train", records=1 << 18, steps=16),
        # thumbnails: small jobs of different scenes in one pool
        dict(name="batch_16", kind="batch", jobs=16, tris=40000, size=192, spp=32, vertices=12),
        # the reference's bidirectional integrator in a closed box
        dict(name="bdpt_512", kind="bdpt", scene="cornell", tris=36, width=512, height=512, spp=8, vertices=10),
        # light tracing: splats from light subpaths
        dict(name="light_720p", kind="light", scene="spheres", tris=1310720, width=1280, height=720, spp=8, vertices=18),
        # loading a scene and showing its first frame: BVH build, allocations
        dict(name="first_frame", kind="first", scene="spheres", tris=1310720, width=640, height=360, spp=1, vertices=10),
        # ray queries from host arrays
        dict(name="trace_1m", kind="trace", scene="spheres", tris=1310720, rays=1 << 20, any=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frame(rng, most):
    """Width, height and spp of at most `most` samples, odd sizes among them."""
    samples = _log(rng, 64 * 64, most)
    spp = _log(rng, 1, min(256, max(1, samples // 4096)))
    pixels = samples / spp
    aspect = rng.uniform(0.6, 2.2)
    width = max(16, int(math.sqrt(pixels * aspect)))
    return width, max(16, int(pixels / width)), spp


def _triangles(rng):
    scene = rng.choice(["cornell", "spheres", "room", "clutter"])
    return scene, 36 if scene == "cornell" else _log(rng, 20000, 1310720)


def draw(rng):
    kind = rng.choice(["nee", "nee", "nee", "nee", "light", "bdpt", "guided", "train", "batch", "first", "trace", "trace"])
    if kind == "train":
        # steps = 0 asks for the gradient alone
        return dict(kind=kind, records=_log(rng, 1000, 1 << 18), steps=rng.choice([0, 0, rng.randint(1, 16)]))
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 24), tris=_log(rng, 10000, 100000), size=_log(rng, 64, 256),
                    spp=_log(rng, 4, 64), vertices=rng.randint(6, 16))
    scene, tris = _triangles(rng)
    if kind == "trace":
        return dict(kind=kind, scene=scene, tris=tris, rays=_log(rng, 1000, 1 << 20), any=rng.random() < 0.5)
    most = {"nee": MOST_SAMPLES / 4, "light": 1280 * 720 * 8, "bdpt": 512 * 512 * 8, "guided": 960 * 540 * 16,
            "first": 640 * 360}[kind]
    width, height, spp = _frame(rng, most)
    case = dict(kind=kind, scene=scene, tris=tris, width=width, height=height, spp=spp, vertices=rng.randint(3, 20))
    if kind == "nee":
        option = rng.choice(["", "", "", "medium", "env"])
        case.update(medium=option == "medium", env=option == "env")
    if kind == "guided":
        case.update(fp8=rng.random() < 0.3)
    return case


# ------------------------------------------------------------------ scenes
def _scene(name, tris, size, seed):
    """A scene of about `tris` triangles; its layout and materials follow the seed."""
    if name == "cornell":
        return scenes.cornell(seed, size)
    if name == "clutter":
        return scenes.cornell_clutter(seed, tris, size)
    level = 5 if tris >= 200_000 else 4 if tris >= 40_000 else 3
    n = max(1, round(tris / (20 * 4 ** level)))
    make = scenes.icospheres if name == "spheres" else scenes.guide_room
    return make(seed, n_spheres=n, level=level, resolution=size)


def _sky(seed):
    """A seeded sky: a gradient, a horizon band and a few bright suns."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:SKY, 0:2 * SKY]
    up = 1.0 - y / SKY
    rgb = np.stack([0.3 + 0.2 * up, 0.35 + 0.3 * up, 0.4 + 0.5 * up], 2)
    for _ in range(3):
        cy, cx, w = rng.uniform(0.1, 0.45) * SKY, rng.uniform(0, 2) * SKY, rng.uniform(2, 8)
        rgb += rng.uniform(20, 200) * np.exp(-((y - cy) ** 2 + (x - cx) ** 2) / (2 * w * w))[:, :, None]
    return rgb.astype(np.float32)


def _case_scene(case, seed):
    sc = _scene(case["scene"], case["tris"], (case.get("width", 64), case.get("height", 64)), seed)
    if case.get("medium"):
        sc = sc.with_medium(sigma_a=0.05, sigma_s=0.4, g=0.7)
    if case.get("env"):
        sc = sc.with_envmap(_sky(seed))
    return sc


def _network(seed):
    """Parameters of a network with 8 different lobes at every vertex: He-normal
    hidden layers, output biases of spread logits, axes and sharpness."""
    rng = np.random.default_rng(seed)
    parts = []
    for l, (k, n) in enumerate(_SHAPES):
        parts.append(rng.normal(scale=math.sqrt(2.0 / k) * (0.3 if l == 4 else 1.0), size=k * n))
        bias = np.zeros(n)
        if l == 4:
            bias = np.column_stack([rng.normal(size=8), rng.normal(size=(8, 3)), rng.uniform(0.5, 6.0, 8)]).ravel()
        parts.append(bias)
    return np.concatenate(parts).astype(np.float32)


def _unit(rng, n):
    v = rng.normal(size=(n, 3))
    return (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)


def _records(case, seed, lo, hi):
    """Training records: points in the scene's box, normals, directions, and
    weights of the long-tailed kind radiance estimates have."""
    rng = np.random.default_rng(seed)
    n = case["records"]
    pos = rng.uniform(lo, hi, size=(n, 3)).astype(np.float32)
    nrm, wo = _unit(rng, n), _unit(rng, n)
    to_light = np.array([0.0, hi[1], 0.0]) - pos + 0.3 * rng.normal(size=(n, 3))
    wi = (to_light / np.linalg.norm(to_light, axis=1, keepdims=True)).astype(np.float32)
    wi = np.where(rng.random((n, 1)) < 0.7, wi, _unit(rng, n))
    return pos, nrm, wo, wi, rng.exponential(size=n).astype(np.float32)


# ------------------------------------------------------------------ a pass
class State:
    """What a program holds between passes."""


def prepare(case, seed):
    s = State()
    s.case, s.seed = case, seed & 0x7FFFFFFF
    s.device = wr.Device(0)
    kind = case["kind"]
    if kind == "train":
        sc = scenes.cornell(seed, (16, 16))
        s.scene = wr.GpuScene(s.device, sc)
        s.guide = wr.Guide(s.scene)
        s.records = _records(case, seed, sc.verts.min(0), sc.verts.max(0))
        s.params = _network(seed)
        s.guide.set_params(s.params)
    elif kind == "batch":
        s.jobs = []
        rng = np.random.default_rng(seed)
        for j in range(case["jobs"]):
            size = int(case["size"] * (1.0 - 0.1 * (j % 4)))
            scene = wr.GpuScene(s.device, scenes.cornell_clutter(seed + j, int(case["tris"] * rng.uniform(0.5, 1.0)), (size, size)))
            s.jobs.append(dict(scene=scene, film=wr.Film(scene), spp=case["spp"], num_path_vertices=case["vertices"],
                               seed=s.seed + j, first_sample=0))
    elif kind == "first":
        s.mesh = _case_scene(case, seed)
    elif kind == "trace":
        sc = _case_scene(case, seed)
        s.scene = wr.GpuScene(s.device, sc)
        half = case["rays"] // 2
        s.rays = np.concatenate([scenes.random_rays(sc, half, seed=seed), scenes.random_rays(sc, case["rays"] - half, seed=seed + 1, inside=True)])
        if case["any"]:  # finite segments, as between two points
            s.rays[:, 7] = np.random.default_rng(seed).uniform(0.1, 20.0, case["rays"]).astype(np.float32)
    else:
        s.scene = wr.GpuScene(s.device, _case_scene(case, seed))
        s.film = wr.Film(s.scene)
        if kind == "guided":
            s.guide = wr.Guide(s.scene)
            s.guide.set_params(_network(seed))
    return s


def _image(film):
    """The finished image as it is written out."""
    return film.image().astype(np.float32)


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "train":
        if case["steps"] == 0:
            loss, grad = s.guide.gradient(*s.records)
            return {"loss": np.float32(loss), "grad": grad}
        s.guide.set_params(s.params)
        loss = s.guide.train(*s.records, steps=case["steps"])
        return {"loss": np.float32(loss), "params": s.guide.get_params()}
    if kind == "batch":
        for j in s.jobs:
            j["film"].clear()
        wr.render_batch(s.jobs)
        return [_image(j["film"]) for j in s.jobs]
    if kind == "trace":
        if case["any"]:
            return {"occluded": s.scene.trace_any(s.rays)}
        geom, prim, t = s.scene.trace_closest(s.rays)
        return {"geom": geom, "prim": prim, "t": t}
    if kind == "first":
        scene = wr.GpuScene(s.device, s.mesh)
        film = wr.Film(scene)
        wr.render_nee(scene, film, case["spp"], num_path_vertices=case["vertices"], seed=s.seed)
        image = _image(film)
        film.close()
        scene.close()
        return image
    s.film.clear()
    common = dict(spp=case["spp"], num_path_vertices=case["vertices"], seed=s.seed)
    if kind == "nee":
        wr.render_nee(s.scene, s.film, **common)
    elif kind == "light":
        wr.render_light(s.scene, s.film, **common)
    elif kind == "bdpt":
        wr.render_bdpt(s.scene, s.film, **common)
    else:
        wr.render_guided(s.scene, s.film, s.guide, guide_fraction=0.4, spp_per_pass=case["spp"], train_steps=0,
                         warmup_passes=0, fp8_inference=case["fp8"], max_guided_bounce=5, **common)
    return _image(s.film)


# ------------------------------------------------------------------ what a pass needs
_SHAPES = [(32, 64), (64, 64), (64, 64), (64, 64), (64, 40)]
_TRI_BYTES = 48 + 2 * 16  # a triangle, and its share of the tree


def work(case):
    """Bytes: scene, rays or records in, images or hits out, once.  Operations:
    per ray, four box tests (12 each) on every level of a 4-wide tree and one
    triangle test (60); per path segment one closest-hit ray, one shadow ray
    and 150 operations of shading; the network's products where it runs."""
    kind = case["kind"]
    if kind == "train":
        n, params = case["records"], sum(k * m for k, m in _SHAPES)
        steps = max(1, case["steps"])
        return {"bytes": 13 * 4.0 * n + 8.0 * params, "flops": 6.0 * n * params * steps}
    tris = case["tris"]
    ray = 48.0 * math.log(max(tris, 5), 4) + 60.0
    if kind == "trace":
        return {"bytes": case["rays"] * (32 + (1 if case["any"] else 12)) + float(_TRI_BYTES * tris), "flops": case["rays"] * ray}
    if kind == "batch":
        samples, pixels, tris = case["jobs"] * 0.73 * case["size"] ** 2 * case["spp"], case["jobs"] * 0.73 * case["size"] ** 2, 0.75 * case["jobs"] * tris
    else:
        pixels = float(case["width"] * case["height"])
        samples = pixels * case["spp"]
    segments = 1 + 0.4 * min(case["vertices"] - 2, 10)  # mean path length
    flops = samples * segments * (2 * ray + 150)
    if kind == "bdpt":
        flops = samples * segments * (2 + segments) * ray
    if kind == "guided":
        flops += samples * min(segments, 5) * 2.0 * sum(k * m for k, m in _SHAPES)
    data = _TRI_BYTES * float(tris) + 12 * pixels
    return {"bytes": data, "flops": flops}


# ------------------------------------------------------------------ 64-bit values
def exact(case, seed):
    """Ray distances by testing every triangle, and the network's gradient, in
    64 bits.  A path tracer's image has none: one rounding sends a path elsewhere."""
    kind = case["kind"]
    if kind == "trace" and not case["any"] and case["scene"] == "cornell":
        return {"geom": None, "prim": None, "t": _exact_t(case, seed)}
    if kind == "train" and case["steps"] == 0:
        return _exact_gradient(case, seed)
    return None


def _exact_t(case, seed):
    sc = _case_scene(case, seed)
    half = case["rays"] // 2
    rays = np.concatenate([scenes.random_rays(sc, half, seed=seed), scenes.random_rays(sc, case["rays"] - half, seed=seed + 1, inside=True)]).astype(np.float64)
    o, tmin, d, tmax = rays[:, 0:3], rays[:, 3], rays[:, 4:7], rays[:, 7]
    best = np.full(len(rays), np.inf)
    v = sc.verts.astype(np.float64)
    for a, b, c in sc.tris:
        e1, e2 = v[b] - v[a], v[c] - v[a]
        p = np.cross(d, e2)
        det = p @ e1
        with np.errstate(divide="ignore", invalid="ignore"):
            q = o - v[a]
            u = (q * p).sum(1) / det
            r = np.cross(q, e1)
            w = (d * r).sum(1) / det
            t = (r @ e2) / det
        hit = (det != 0) & (u >= 0) & (w >= 0) & (u + w <= 1) & (t > tmin) & (t <= tmax) & (t < best)
        best = np.where(hit, t, best)
    return best


def _oct(d):
    r = np.abs(d).sum(1)
    u, v = d[:, 0] / r, d[:, 2] / r
    low, one = d[:, 1] < 0, lambda x: np.where(x >= 0, 1.0, -1.0)
    return [np.clip(0.5 * x + 0.5, 0, 1) for x in (np.where(low, (1 - abs(v)) * one(u), u), np.where(low, (1 - abs(u)) * one(v), v))]


def _exact_gradient(case, seed):
    """Mean over the records of -w log q(wi), q the mixture of 8 von Mises-Fisher
    lobes the network gives, and its gradient."""
    sc = scenes.cornell(seed, (16, 16))
    lo, hi = sc.verts.min(0).astype(np.float64), sc.verts.max(0).astype(np.float64)
    pos, nrm, wo, wi, weight = (a.astype(np.float64) for a in _records(case, seed, sc.verts.min(0), sc.verts.max(0)))
    params = _network(seed).astype(np.float64)
    layers, at = [], 0
    for k, n in _SHAPES:
        layers.append((params[at:at + k * n].reshape(k, n), params[at + k * n:at + k * n + n]))
        at += k * n + n
    total, grads = 0.0, [(np.zeros_like(w), np.zeros_like(b)) for w, b in layers]
    for at in range(0, len(pos), 32768):
        part = slice(at, at + 32768)
        code = [*np.clip((pos[part] - lo) / (hi - lo), 0, 1).T, *_oct(nrm[part]), *_oct(wo[part])]
        x = np.concatenate([np.exp(-0.5 * ((c[:, None] - (np.arange(k) + 0.5) / k) * k) ** 2)
                            for c, k in zip(code, (6, 6, 6, 4, 4, 3, 3))], 1)
        ins = []
        for l, (w, b) in enumerate(layers):
            ins.append(x)
            x = x @ w + b
            if l < 4:
                x = np.maximum(x, 0)
        o = x.reshape(-1, 8, 5)
        scale = weight[part, None] / len(pos)
        m = o[:, :, 0].max(1, keepdims=True)
        logw = o[:, :, 0] - m - np.log(np.exp(o[:, :, 0] - m).sum(1, keepdims=True))
        size = np.linalg.norm(o[:, :, 1:4], axis=2, keepdims=True)
        mu = o[:, :, 1:4] / size
        raw = np.logaddexp(0, o[:, :, 4])
        lam = np.clip(raw, 0.05, 2000.0)
        cos = (mu * wi[part, None]).sum(2)
        logc = logw + np.log(lam / (2 * np.pi)) - np.log(-np.expm1(-2 * lam)) + lam * (cos - 1)
        logq = np.logaddexp.reduce(logc, axis=1, keepdims=True)
        share = np.exp(logc - logq)
        total += float(-(scale * logq).sum())
        g = np.empty_like(o)
        g[:, :, 0] = -scale * (share - np.exp(logw))
        dmu = (share * lam)[:, :, None] * wi[part, None]
        g[:, :, 1:4] = -scale[:, :, None] * (dmu - mu * (mu * dmu).sum(2, keepdims=True)) / size
        inside = (raw > 0.05) & (raw < 2000.0)
        with np.errstate(over="ignore"):
            dlam = 1 / lam - 2 / np.expm1(2 * lam) + cos - 1
        g[:, :, 4] = -scale * share * dlam * np.where(inside, 1 / (1 + np.exp(-o[:, :, 4])), 0)
        dy = g.reshape(-1, 40)
        for l in range(4, -1, -1):
            grads[l][0][...] += ins[l].T @ dy
            grads[l][1][...] += dy.sum(0)
            if l:
                dy = (dy @ layers[l][0].T) * (ins[l] > 0)
    return {"loss": total, "grad": np.concatenate([np.concatenate([w.ravel(), b]) for w, b in grads])}
