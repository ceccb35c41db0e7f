"""Performance cases: the work a program has this library do, one pass each.

Every case goes through the public entry points (globillum_amd.context.Context,
globillum_amd.diff, and the gi_trace_*_device calls of include/gi_hip.h) with
scenes of the package's own generators.  Kinds:

  closest, any   trace_closest / trace_any on host arrays (the tracer plugin's calls)
  closest_dev    gi_trace_closest_device on rays that already lie on the GPU
  render         Context.render, then every view's image on the host
  progress       progress_begin, then one sample per pixel and the image, step by step
  grad           differentiable render through torch autograd (materials, emission)
  texgrad        render, adjoint, per-texel gradient of an instanced, textured scene
  scene          a new scene: upload, device BVH build, first trace

listed() names them, draw() takes others of the same ranges, prepare() makes
a case's inputs, run() is one pass, work() its least bytes and operations and
exact() its result in 64 bits where that can be had.
"""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import math

import numpy as np
import torch

from globillum_amd import diff, scenes
from globillum_amd._lib import (FLAG_BATCHED, FLAG_GRAPH, FLAG_PHONG, FLAG_PIXEL_CENTRE, HIT)
from globillum_amd.context import Context

FLT_MAX = float(np.finfo(np.float32).max)


def listed():
    return [
        # picking and probes: a thousand rays, one call, latency is all there is
        dict(name="pick_1k", kind="closest", scene="cornell", rays=1024),
        # the plugin's any-hit tracer on host arrays: shadow rays of one tile, two-level scene, odd count
        dict(name="shadow_host_250k", kind="any", scene="instanced", cells=64, spheres=200, rays=249_983),
        # a renderer that keeps its rays on the GPU: one bounce wave of a 1280x800 image
        dict(name="bounce_dev_1m", kind="closest_dev", scene="terrain", cells=256, spheres=1000, rays=1_024_000),
        # the small configuration: 34-triangle Cornell box, captured graph
        dict(name="render_cornell_256", kind="render", scene="cornell", w=256, h=256, spp=16, depth=4, rr=0,
             views=1, flags=FLAG_BATCHED | FLAG_GRAPH),
        # sky and rect light through a thin lens, one view at a time, odd sizes (a plugin frame with its options)
        dict(name="render_sky_lens", kind="render", scene="sky", w=641, h=477, spp=9, depth=5, rr=3, views=1, flags=0),
        # 16 views of uneven size and sample count with Russian roulette in one captured loop
        dict(name="render_views_16", kind="render", scene="views", w=0, h=0, spp=0, depth=8, rr=3, views=16,
             flags=FLAG_BATCHED | FLAG_GRAPH),
        # the ~300k-triangle configuration
        dict(name="render_terrain_720p", kind="render", scene="terrain", cells=256, spheres=1000, mats=32, lights=4,
             w=1280, h=720, spp=64, depth=8, rr=0, views=1, flags=FLAG_BATCHED),
        # the large combined configuration, 4.2M triangles, instances, texture, 64 lights, four 4K views
        dict(name="render_large_4k_x4", kind="render", scene="large", cells=2048, spheres=2000, mats=256, lights=64,
             w=3840, h=2160, spp=16, depth=6, rr=0, views=4, flags=FLAG_BATCHED),
        # an interactive viewer: one sample per pixel a step, the image shown after each
        dict(name="progress_640", kind="progress", scene="textured", w=640, h=480, depth=4, steps=4),
        # inverse rendering, the 108k-triangle differentiation configuration, through torch autograd
        dict(name="grad_diff_512", kind="grad", scene="diff", cells=200, spheres=50, mats=64, lights=4, w=512, h=512,
             spp=16, depth=4),
        # material, light and per-texel gradients of an instanced scene
        dict(name="texgrad_720p", kind="texgrad", scene="large", cells=512, spheres=500, mats=64, lights=16, w=1280,
             h=720, spp=16, depth=6, views=1, tex=1024),
        # geometry that changes: upload, device SAH build, first trace
        dict(name="scene_sah_291k", kind="scene", scene="terrain", cells=256, spheres=1000, mats=32, lights=4,
             builder="sah", rays=65_537),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "any", "closest_dev", "render", "render", "render", "progress", "grad", "texgrad",
                       "scene"])
    if kind == "closest":
        sc = rng.choice(["cornell", "terrain"])
        c = dict(kind=kind, scene=sc, rays=_log(rng, 256, 300_000))
        if sc == "terrain":
            c.update(cells=_log(rng, 16, 256), spheres=_log(rng, 4, 300))
        return c
    if kind == "any":
        return dict(kind=kind, scene="instanced", cells=_log(rng, 8, 128), spheres=_log(rng, 10, 400),
                    rays=_log(rng, 1000, 500_000))
    if kind == "closest_dev":
        return dict(kind=kind, scene="terrain", cells=_log(rng, 16, 512), spheres=_log(rng, 4, 1000),
                    rays=_log(rng, 20_000, 4_000_000))
    if kind == "render":
        sc = rng.choice(["cornell", "sky", "views", "terrain", "large"])
        flags = rng.choice([0, FLAG_BATCHED, FLAG_BATCHED | FLAG_GRAPH])
        w = _log(rng, 64, 1920)
        h = max(32, int(w * rng.uniform(0.4, 1.1)))
        c = dict(kind=kind, scene=sc, w=w, h=h, spp=_log(rng, 1, 64), depth=rng.randint(2, 8),
                 rr=rng.choice([0, 0, 3]), views=1, flags=flags)
        if sc == "cornell" and rng.random() < 0.3:
            c["flags"] |= rng.choice([FLAG_PHONG, FLAG_PIXEL_CENTRE])
        if sc == "views":
            c.update(w=0, h=0, spp=0, views=rng.randint(2, 16))
        if sc == "terrain":
            c.update(cells=_log(rng, 16, 400), spheres=_log(rng, 4, 1000), mats=rng.randint(4, 64),
                     lights=rng.randint(1, 16))
        if sc == "large":
            c.update(cells=2 * _log(rng, 32, 700), spheres=_log(rng, 10, 2000), mats=rng.randint(8, 256),
                     lights=rng.randint(1, 64), views=rng.randint(1, 3))
        c["spp"] = max(1, min(c["spp"], 120_000_000 // max(1, w * h * c["views"])))
        return c
    if kind == "progress":
        w = _log(rng, 64, 1280)
        return dict(kind=kind, scene="textured", w=w, h=max(32, int(w * rng.uniform(0.5, 1.0))),
                    depth=rng.randint(2, 8), steps=rng.randint(1, 8))
    if kind == "grad":
        w = _log(rng, 64, 700)
        return dict(kind=kind, scene="diff", cells=_log(rng, 16, 250), spheres=_log(rng, 4, 100),
                    mats=rng.randint(4, 96), lights=rng.randint(1, 9), w=w, h=max(32, int(w * rng.uniform(0.5, 1.1))),
                    spp=_log(rng, 1, 24), depth=rng.randint(2, 6))
    if kind == "texgrad":
        w = _log(rng, 96, 1280)
        return dict(kind=kind, scene="large", cells=2 * _log(rng, 16, 300), spheres=_log(rng, 10, 600),
                    mats=rng.randint(8, 128), lights=rng.randint(1, 32), w=w, h=max(64, int(w * rng.uniform(0.4, 0.7))),
                    spp=_log(rng, 1, 16), depth=rng.randint(2, 6), views=1, tex=_log(rng, 60, 1100))
    return dict(kind="scene", scene="terrain", cells=_log(rng, 16, 600), spheres=_log(rng, 4, 600),
                mats=rng.randint(4, 64), lights=rng.randint(1, 8),
                builder=rng.choice(["sah", "sah", "device", "ploc"]), rays=_log(rng, 1000, 200_000))


# ------------------------------------------------------------------ scenes --
@functools.lru_cache(maxsize=1)
def _large(cells, spheres, mats, lights, w, h, spp, depth, views, tex):
    """The large scenes' geometry: an asset, made once (seconds of numpy);
    cameras and materials are the seed's."""
    return scenes.large_combined(cells=(cells, cells // 2), n_spheres=spheres, n_mats=mats, n_lights=lights, w=w, h=h,
                                 spp=spp, depth=depth, n_views=views, texture=(tex, tex))


def _scene(c, seed):
    """The case's scene: geometry, cameras and materials follow the seed (the
    large scenes' geometry does not)."""
    k = c["scene"]
    if k == "cornell":
        sc = scenes.cornell_boxes(seed=seed, w=c.get("w", 64), h=c.get("h", 64), spp=c.get("spp", 1),
                                  depth=c.get("depth", 4))
    elif k == "sky":
        sc = scenes.sky_scene(w=c["w"], h=c["h"], spp=c["spp"], depth=c["depth"], seed=seed)
        sc.views["aperture"], sc.views["focus_distance"] = 0.15, 10.0
    elif k == "views":
        # image sizes and sample counts are the workload (fixed by the view
        # count); the cameras follow the seed
        sc = scenes.cornell_batch(seed=3, n_views=c["views"], depth=c["depth"])
        other = scenes.cornell_batch(seed=1000 + seed, n_views=c["views"], depth=c["depth"])
        for f in ("pos", "dir", "fovy"):
            sc.views[f] = other.views[f]
    elif k == "terrain":
        sc = scenes.terrain_spheres(seed=seed, cells=(c["cells"], c["cells"]), n_spheres=c["spheres"],
                                    n_mats=c.get("mats", 32), n_lights=c.get("lights", 4), w=c.get("w", 64),
                                    h=c.get("h", 64), spp=c.get("spp", 1), depth=c.get("depth", 4))
    elif k == "instanced":
        sc = scenes.instanced_terrain(seed=seed, cells=(c["cells"], c["cells"]), n_instances=c["spheres"])
    elif k == "textured":
        sc = scenes.textured_scene(seed=seed, w=c["w"], h=c["h"], spp=c["steps"], depth=c["depth"])
    elif k == "diff":
        sc = scenes.diff_scene(seed=seed, cells=(c["cells"], c["cells"] * 5 // 4), n_spheres=c["spheres"],
                               n_mats=c["mats"], n_lights=c["lights"], w=c["w"], h=c["h"], spp=c["spp"],
                               depth=c["depth"])
    else:
        sc = _large(c["cells"], c["spheres"], c["mats"], c["lights"], c["w"], c["h"], c["spp"], c["depth"],
                    c["views"], c.get("tex", 1024))
        rng = np.random.default_rng(seed)
        sc = dataclasses.replace(sc, mats=sc.mats.copy(), views=sc.views.copy(), opts=sc.opts.copy())
        sc.views["pos"] += rng.uniform(-3.0, 3.0, sc.views["pos"].shape).astype(np.float32)
        sc.mats["color"] = rng.uniform(0.0, 1.0, sc.mats["color"].shape)
        sc.mats["roughness"] = rng.uniform(0.05, 1.0, len(sc.mats))
    if "flags" in c:
        sc.opts["flags"] = c["flags"]
        sc.opts["rr_start"] = c["rr"]
    sc.opts["seed"] = seed % 97
    return sc


def _rays(c, sc, seed):
    """Rays of the case: (orig, dir, max_t), float32."""
    rng = np.random.default_rng(1_000_003 * (seed + 1))
    n = c["rays"]
    if c["kind"] in ("closest", "scene"):
        # pinhole rays of the scene's camera in pixel order, jittered in the pixel
        v = sc.views[0]
        w = max(1, int(math.sqrt(n * 1.3)))
        h = -(-n // w)
        i = np.arange(n)
        W = v["dir"].astype(np.float64)
        U = np.cross(v["up"].astype(np.float64), W)
        U /= np.linalg.norm(U)
        V = np.cross(W, U)
        half = math.tan(math.radians(float(v["fovy"]) / 2))
        x = ((i % w + rng.random(n)) / w * 2 - 1) * half
        y = ((i // w + rng.random(n)) / h * 2 - 1) * half
        d = W + x[:, None] * U + y[:, None] * V
        o = np.broadcast_to(v["pos"].astype(np.float64), d.shape)
        t = np.full(n, FLT_MAX, np.float32)
        return (np.ascontiguousarray(o, np.float32),
                (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32), t)
    # surface points in triangle order, as a renderer's compacted queue holds neighbours
    k = np.sort(rng.integers(0, len(sc.tris), n))
    b = rng.random((n, 2))
    f = b.sum(1) > 1
    b[f] = 1 - b[f]
    a, e1, e2 = (sc.tris[q][k].astype(np.float64) for q in ("a", "b", "c"))
    p = a + b[:, :1] * (e1 - a) + b[:, 1:] * (e2 - a)
    nrm = sc.tris["na"][k].astype(np.float64)
    o = p + 1e-3 * nrm
    if c["kind"] == "any":  # towards a point of a random light
        lt = sc.lights[rng.integers(0, len(sc.lights), n)]
        q = lt["center"].astype(np.float64)
        q[:, 0] += (rng.random(n) - 0.5) * lt["wh"][:, 0]
        q[:, 2] += (rng.random(n) - 0.5) * lt["wh"][:, 1]
        d = q - o
        t = np.linalg.norm(d, axis=1)
        return o.astype(np.float32), (d / t[:, None]).astype(np.float32), t.astype(np.float32)
    d = rng.normal(size=(n, 3))  # cosine distributed about the normal
    d = nrm + d / np.linalg.norm(d, axis=1, keepdims=True)
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-6)
    return o.astype(np.float32), d.astype(np.float32), np.full(n, FLT_MAX, np.float32)


# ----------------------------------------------------------- prepare and run --
def prepare(case, seed):
    c = case
    sc = _scene(c, seed)
    s = dict(c=c, scene=sc)
    ctx = s["ctx"] = Context(0)
    if c["kind"] == "scene":
        s["rays"] = _rays(c, sc, seed)
        return s
    ctx.upload(sc, builder="sah")
    if c["kind"] in ("closest", "any"):
        s["rays"] = _rays(c, sc, seed)
    elif c["kind"] == "closest_dev":
        s["rays"] = [torch.from_numpy(a).cuda() for a in _rays(c, sc, seed)]
        s["hits"] = torch.empty((c["rays"], 4), dtype=torch.float32, device="cuda")
    elif c["kind"] == "grad":
        g = torch.Generator().manual_seed(seed)
        s["mats"] = torch.from_numpy(diff.material_params(sc)).cuda()
        s["emission"] = torch.from_numpy(sc.lights["col"].copy()).cuda()
        s["target"] = (0.5 * torch.rand((c["w"] * c["h"], 3), generator=g)).cuda()
    elif c["kind"] == "texgrad":
        rng = np.random.default_rng(seed)
        s["dl"] = rng.normal(0.0, 1.0 / (c["w"] * c["h"]), (c["views"] * c["w"] * c["h"], 3)).astype(np.float32)
    return s


def _hits(h):
    return {"t": h["t"], "beta": h["beta"], "gamma": h["gamma"], "ref": h["ref"].view(np.int32)}


def _dev(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    c, ctx, sc = state["c"], state["ctx"], state["scene"]
    kind = c["kind"]
    if kind == "closest":
        return _hits(ctx.trace_closest(*state["rays"]))
    if kind == "any":
        return ctx.trace_any(*state["rays"])
    if kind == "closest_dev":
        o, d, t = state["rays"]
        out = state["hits"]
        ctx._ck(ctx.lib.gi_trace_closest_device(ctx.h, _dev(o), _dev(d), _dev(t), c["rays"], _dev(out)))
        return {"t_beta_gamma": out[:, :3], "ref": out[:, 3].view(torch.int32)}
    if kind == "render":
        return ctx.render().images()
    if kind == "progress":
        ctx.progress_begin()
        imgs, done = [], False
        while not done:
            done = ctx.progress_step()
            imgs.append(ctx.image(0))
        return imgs
    if kind == "grad":
        m = state["mats"].clone().requires_grad_(True)
        e = state["emission"].clone().requires_grad_(True)
        img = diff.render(ctx, m, e)
        ((img - state["target"]) ** 2).mean().backward()
        return {"image": img.detach(), "d_mats": m.grad, "d_emission": e.grad}
    if kind == "texgrad":
        imgs = ctx.render().images()
        g, de = ctx.adjoint(state["dl"])
        return {"images": imgs, "d_mats": g, "d_emission": de, "d_texels": ctx.texture_grad(0)}
    ctx.upload(sc, builder=c["builder"])
    return _hits(ctx.trace_closest(*state["rays"]))


# --------------------------------------------------------------------- work --
def _tris(c):
    """(triangles in memory, triangles a ray can meet)."""
    k = c["scene"]
    if k == "cornell" or k == "views":
        return 34, 34
    if k == "sky":
        return 210, 210
    if k == "textured":
        return 2048 + 216, 2048 + 40 * 216
    if k == "instanced":
        n = 2 * c["cells"] ** 2
        return n + 220, n + 73 * c["spheres"]
    if k == "large":
        n = c["cells"] ** 2
        return n + 160, n + 160 * c["spheres"]
    n = 2 * c["cells"] ** 2 * (5 if k == "diff" else 4) // 4
    return n + 160 * c["spheres"], n + 160 * c["spheres"]


def _samples(c):
    """(pixels, samples) of a render."""
    if c["scene"] == "views":
        v = scenes.cornell_batch(seed=3, n_views=c["views"], depth=c["depth"]).views
        px = v["w"].astype(np.int64) * v["h"]
        return int(px.sum()), int((px * v["spp"]).sum())
    px = c["w"] * c["h"] * c.get("views", 1)
    return px, px * c.get("spp", c.get("steps", 1))


def work(case):
    """Least work of one pass: the scene's vertices (36 B), normals and texture
    coordinates (64 B) read once where shading needs them, rays and results or
    images once; operations: per ray two box tests (24 flops) a level of a
    binary tree and four triangle tests (60), 500 per shaded vertex."""
    c = case
    mem, met = _tris(c)
    per_ray = 2 * 24 * math.log2(max(2, met)) + 4 * 60
    if c["kind"] in ("closest", "any", "closest_dev", "scene"):
        n = c["rays"]
        b = 36.0 * mem + n * (28 + (1 if c["kind"] == "any" else 16))
        f = n * per_ray
        if c["kind"] == "scene":  # the uploaded records once; binning, 3 axes a level
            b += 64.0 * mem
            f += 20.0 * mem * math.log2(max(2, mem))
        return {"bytes": b, "flops": f}
    px, samples = _samples(c)
    depth = c["depth"]
    # Russian roulette ends paths early: about half of their later vertices
    verts = samples * (depth if not c.get("rr") else min(depth, c["rr"] + (depth - c["rr"]) / 2))
    f = verts * (2 * per_ray + 500)
    b = 100.0 * mem + 12.0 * px * (c["steps"] if c["kind"] == "progress" else 1)
    if c["kind"] in ("grad", "texgrad"):  # forward, and its adjoint: shading and its derivative once more
        f += verts * 1500
        b += 12.0 * px + (12.0 * c["tex"] ** 2 if c["kind"] == "texgrad" else 0)
    return {"bytes": b, "flops": f}


# -------------------------------------------------------------------- exact --
def exact(case, seed):
    """Closest hits in 64 bits by testing every triangle; other results are
    whole numbers or random walks whose every turn depends on the last bits."""
    c = case
    if c["kind"] not in ("closest", "scene") or c["rays"] * _tris(c)[0] > 25e9:
        return None
    sc = _scene(c, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    o, d, mt = (torch.from_numpy(a).to(dev).double() for a in _rays(c, sc, seed))
    a = torch.from_numpy(sc.tris["a"].copy()).to(dev).double()
    e1 = torch.from_numpy(sc.tris["b"].copy()).to(dev).double() - a
    e2 = torch.from_numpy(sc.tris["c"].copy()).to(dev).double() - a
    n = len(o)
    out = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    out[:, 0] = FLT_MAX
    step = max(1, int(3e8) // len(a))
    ng = torch.linalg.cross(e1, e2)
    for i in range(0, n, step):
        O, D = o[i:i + step], d[i:i + step]
        # Cramer's rule on a + b e1 + g e2 = O + t D, products over (rays, triangles)
        det = -(D @ ng.T)
        # (O - a) x e2 . D and D . (e1 x (O - a)) expanded into matrix products
        ca = torch.linalg.cross(O, D)
        u = ca @ e2.T + D @ torch.linalg.cross(a, e2).T
        v = -(ca @ e1.T) - D @ torch.linalg.cross(a, e1).T
        t = O @ ng.T - (a * ng).sum(1)
        u, v, t = u / det, v / det, t / det
        ok = (det != 0) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0) & (t <= mt[i:i + step, None])
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, k = t.min(1)
        hit = torch.isfinite(best)
        r = torch.arange(len(O), device=dev)
        vals = torch.stack([best, u[r, k], v[r, k]], 1)
        out[i:i + step][hit] = vals[hit]
    x = out.cpu().numpy()
    return {"t": x[:, 0], "beta": x[:, 1], "gamma": x[:, 2], "ref": None}


assert HIT.itemsize == 16
