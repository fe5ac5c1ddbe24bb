"""Workloads a renderer built on illume_amd runs: whole calls through the public entry points
(Context.render, render_noalloc, render_batch, submit/wait/result), each with the scene resident
in HBM and the image returned to the caller as the binding returns it.

    listed()             the named workloads
    draw(rng)            one more workload of the same ranges
    prepare(case, seed)  the context, scenes and render parameters a program holds before the call
    run(state)           one call, its images and its segment count
    work(case)           bytes and operations of one call that no implementation can do without
    exact(case, seed)    the Cornell box images in 64-bit arithmetic, by brute force over triangles

A seed changes the geometry (noise of the displaced meshes, turn of the Cornell boxes), the
camera's position and the index of the first sample.
"""
import functools
import math

import numpy as np
import torch

import illume_amd
from illume_amd import scenes as S
from illume_amd._abi import render_params

MAX_PATHS = 1280 * 720 * 64     # the largest listed image, in samples

# Per scene family: mean closest-hit queries per path at the family's depth, child-box tests and
# triangle tests per query of an ordered walk, rounded (counted by the renderer's own test counters).
COUNTS = {"box": (4.6, 13.7, 2.2), "materials": (2.6, 33.0, 2.8), "metal": (2.3, 17.0, 2.3),
          "subsurface": (5.7, 40.0, 2.6), "instances": (3.0, 70.0, 5.2)}
BOX_FLOPS, TRI_FLOPS, SHADE_FLOPS = 12.0, 30.0, 150.0


# ---------------------------------------------------------------- scenes

@functools.lru_cache(maxsize=8)
def _sphere(n):
    """Geodesic sphere of 20 n^2 triangles: unit vertices and indices."""
    return S.icosphere(n)


@functools.lru_cache(maxsize=1)
def _sky():
    return S.sky_env(2048, 1024)


def _bumpy(n, seed):
    """The displaced sphere of the benchmark scenes, its noise from the seed."""
    v, t = _sphere(n)
    noise = (S.value_noise(v * 3.0, seed) + 0.5 * S.value_noise(v * 6.0, seed + 101)
             + 0.25 * S.value_noise(v * 12.0, seed + 202)) / 1.75
    return dict(positions=(v * (1.0 + 0.1 * noise)[:, None]).astype(np.float32), indices=t,
                face_normals=True, leaf_size=4)


def _spec(kind, detail, seed):
    """A scene of the family with 20 detail^2 triangles per mesh (the Cornell box has 36)."""
    rng = np.random.RandomState(seed & 0x7FFFFFFF)
    nseed = int(rng.randint(1, 1 << 20))
    if kind == "box":
        spec, _ = S.cornell()
        for i in (6, 7):
            spec["instances"][i]["transform"]["rotation"] = [0.0, float(np.float32(rng.uniform(-40, 40))), 0.0]
    elif kind == "materials":
        spec, _ = S.tiny_mesh_scene(n=1)
        v, t = _sphere(detail)
        spec["meshes"][0] = dict(positions=v.astype(np.float32), indices=t, normals=v.astype(np.float32),
                                 face_normals=False, leaf_size=4)
        for i in spec["instances"][:9]:
            i["transform"]["rotation"] = [float(np.float32(x)) for x in rng.uniform(-60, 60, 3)]
    elif kind == "metal":
        spec, _ = S.gold_spheres(n=1)
        spec["meshes"][0] = _bumpy(detail, nseed)
    elif kind == "subsurface":
        spec, _ = S.subsurface(n=1, env_size=(8, 4))
        spec["meshes"][0] = _bumpy(detail, nseed)
        spec["environment"] = dict(type="bitmap", texels=_sky())
    else:
        spec, _ = S.instanced(n=1)
        spec["meshes"][0] = _bumpy(detail, nseed)
    cam = spec["camera"]["transform"]
    cam["translation"] = [float(np.float32(c + d)) for c, d in zip(cam["translation"], rng.uniform(-0.05, 0.05, 3))]
    return spec


TONEMAP = {"box": "linear", "materials": "reinhard", "metal": "linear", "subsurface": "filmic",
           "instances": "uncharted"}

# Requests of the batched and served workloads, as (scene, share of the width and height, share of
# the samples): users ask for different scenes at different sizes at the same time.
MIX = [("metal", 1.0, 0.25), ("subsurface", 0.5, 0.5), ("box", 1.0, 1.0), ("instances", 0.75, 0.25),
       ("metal", 0.25, 1.0), ("box", 0.5, 0.5), ("subsurface", 0.75, 0.25), ("instances", 0.5, 0.5),
       ("metal", 0.5, 0.5), ("box", 0.25, 1.0), ("subsurface", 0.25, 1.0), ("instances", 0.25, 0.75)]


def _requests(case):
    """(scene family, width, height, spp, depth) of each request of the call."""
    w, h, spp, depth = case["width"], case["height"], case["spp"], case["depth"]
    if case["form"] in ("render", "noalloc"):
        return [(case["scene"], w, h, spp, depth)]
    return [(k, max(1, int(w * s)), max(1, int(h * s)), max(1, int(spp * f)), depth)
            for k, s, f in MIX[:case["requests"]]]


def _case(form, scene, detail, width, height, spp, depth, layout, tri="mt", requests=1, name=None):
    c = dict(form=form, scene=scene, detail=detail, width=width, height=height, spp=spp, depth=depth,
             layout=layout, tri=tri, requests=requests)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a material preview or a unit test: the smallest image, one sample, all of it latency
        _case("render", "box", 1, 64, 64, 1, 8, "fp32", name="preview 64x64"),
        # the Cornell box of the benchmark's configuration 0, at the library's default settings
        _case("render", "box", 1, 256, 256, 16, 8, "fp32", name="cornell 256x256"),
        # an interactive viewer's pass: one sample per pixel of a full-HD image, again and again
        _case("render", "metal", 71, 1920, 1080, 1, 16, "quant8", name="viewer pass 1080p"),
        # every material, smooth normals, a textured sky; an odd-sized image and sample count
        _case("render", "materials", 16, 333, 251, 7, 12, "fp32", name="materials 333x251"),
        # the headline benchmark: 100,820 triangles, 1024x1024, 64 spp, depth 16
        _case("render", "metal", 71, 1024, 1024, 64, 16, "quant8", name="metal 1024x1024"),
        # the same scene at the default node layout with the watertight triangle test
        _case("render", "metal", 71, 640, 480, 32, 16, "fp32", tri="watertight", name="metal watertight 640x480"),
        # subsurface scattering, long paths (configuration 2: 524,880 triangles, depth 45)
        _case("render", "subsurface", 162, 960, 720, 32, 45, "quant8", name="subsurface 960x720"),
        # the same material on a small mesh and image: long paths, short queues
        _case("render", "subsurface", 40, 320, 240, 8, 45, "fp32", name="subsurface 320x240"),
        # 12 instances of a 722,000-triangle mesh, a final-quality 720p frame
        _case("render", "instances", 190, 1280, 720, 64, 16, "quant8", name="instances 1280x720"),
        # a caller that may not allocate device memory (tight serving loop)
        _case("noalloc", "metal", 40, 400, 300, 8, 16, "quant8", name="noalloc 400x300"),
        # a batch of requests over four scenes in one call
        _case("batch", "mix", 48, 512, 512, 48, 16, "quant8", requests=12, name="batch of 12"),
        # requests that arrive together at a server
        _case("served", "mix", 48, 640, 360, 32, 16, "fp32", requests=8, name="served 8"),
    ]


def _cost(case):
    """Work of a case in the largest listed image's samples, queries and box tests weighted in."""
    t = 0.0
    for k, w, h, spp, depth in _requests(case):
        q, b, _ = COUNTS[k]
        t += w * h * spp * q * (b + 15.0)
    q, b, _ = COUNTS["instances"]
    return t / (MAX_PATHS * q * (b + 15.0))


def draw(rng):
    while True:
        form = rng.choice(["render"] * 6 + ["noalloc", "batch", "served", "served"])
        many = form in ("batch", "served")
        scene = "mix" if many else rng.choice(["box", "materials", "metal", "subsurface", "instances"])
        detail = int(round(math.exp(rng.uniform(math.log(4), math.log(64 if many else 190)))))
        if scene == "box":
            detail = 1
        px = math.exp(rng.uniform(math.log(48 * 48), math.log(640 * 360 if many else 1920 * 1080)))
        aspect = math.exp(rng.uniform(math.log(0.6), math.log(2.2)))
        width = max(16, int(math.sqrt(px * aspect)))
        height = max(16, int(px / width))
        spp = int(round(math.exp(rng.uniform(0.0, math.log(64)))))
        depth = rng.randint(32, 45) if scene == "subsurface" else rng.randint(8, 24)
        case = _case(form, scene, detail, width, height, spp, depth, rng.choice(["fp32", "quant8"]),
                     tri=rng.choice(["mt", "mt", "mt", "watertight"]),
                     requests=rng.randint(3, 12) if many else 1)
        if _cost(case) <= 0.9 and (form != "noalloc" or width * height <= 1 << 20):
            return case


# ---------------------------------------------------------------- the call

def prepare(case, seed):
    ctx = illume_amd.Context(0, bvh_layout=case["layout"], tri_test=case["tri"])
    reqs = _requests(case)
    rng = np.random.RandomState((seed + 7) & 0x7FFFFFFF)
    first = int(rng.randint(0, 1 << 16))
    scenes = {}
    for k, _, _, _, _ in reqs:
        if k not in scenes:
            scenes[k] = ctx.scene(_spec(k, case["detail"], seed))
    params = [render_params(w, h, spp, depth, ray_bias=1e-4, tonemap=TONEMAP[k], first_sample=first)
              for k, w, h, spp, depth in reqs]
    return dict(form=case["form"], ctx=ctx, scenes=[scenes[r[0]] for r in reqs], params=params)


def _image(acc, pix):
    return {"sum": acc, "pixels": pix.view(np.int64)}


def run(state):
    ctx, form = state["ctx"], state["form"]
    if form == "served":
        reqs = [ctx.submit(s, p) for s, p in zip(state["scenes"], state["params"])]
        images = []
        for r in reqs:
            r.wait()
            images.append(_image(*r.result()))
            r.free()
        return {"images": images}
    if form == "batch":
        images, info = ctx.render_batch(state["scenes"], state["params"])
        return {"images": [_image(*i) for i in images], "segments": info["segments"]}
    call = ctx.render if form == "render" else ctx.render_noalloc
    acc, pix, info = call(state["scenes"][0], state["params"][0])
    return {"images": [_image(acc, pix)], "segments": info["segments"]}


def work(case):
    """Scenes read once, images written once (12 B of sums and 24 B of pixel each); the operations
    of the family's mean number of closest-hit queries, box and triangle tests and shading steps."""
    nbytes = flops = 0.0
    seen = set()
    for k, w, h, spp, _ in _requests(case):
        q, b, t = COUNTS[k]
        nbytes += 36.0 * w * h
        flops += w * h * spp * q * (b * BOX_FLOPS + t * TRI_FLOPS + SHADE_FLOPS)
        if k not in seen:
            seen.add(k)
            nbytes += 36 * 36 if k == "box" else 20 * case["detail"] ** 2 * 36
            nbytes += 2048 * 1024 * 16 if k == "subsurface" else 0
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------- 64-bit Cornell box

_M32 = 0xFFFFFFFF


def _shr(x, n):
    """Logical right shift of 64-bit patterns held in int64."""
    return (x >> n) & ((1 << (64 - n)) - 1)


def _s64(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


class _Pcg:
    """PCG32 (XSH-RR, 64-bit state) of every path at once."""
    MULT = _s64(6364136223846793005)

    def __init__(self, passes, pixels):
        self.inc = (pixels << 1) | 1
        self.s = torch.zeros_like(pixels)
        self.next()
        self.s = self.s + passes
        self.next()

    def next(self):
        old = self.s
        self.s = old * self.MULT + self.inc
        x = _shr(_shr(old, 18) ^ old, 27) & _M32
        r = _shr(old, 59)
        return ((x >> r) | (x << ((32 - r) & 31))) & _M32

    def uniform(self):
        return ((self.next() >> 8) + 1).double() * 2.0 ** -24


def _wang(a):
    a = (a ^ 61) ^ (a >> 16)
    a = (a + (a << 3)) & _M32
    a = a ^ (a >> 4)
    a = (a * 0x27D4EB2D) & _M32
    return a ^ (a >> 15)


def _matrix(t):
    f = lambda v: [float(np.float32(x)) for x in v]  # noqa: E731
    m = np.eye(4)
    for axis, deg in zip(range(3), f(t.get("rotation", [0, 0, 0]))):
        c, s = math.cos(math.radians(deg)), math.sin(math.radians(deg))
        r = np.eye(4)
        i, j = [(1, 2), (2, 0), (0, 1)][axis]
        r[i, i] = r[j, j] = c
        r[i, j], r[j, i] = -s, s
        m = m @ r
    tr = np.eye(4)
    tr[:3, 3] = f(t["translation"])
    return tr @ m @ np.diag(f(t.get("scale", [1, 1, 1])) + [1.0])


def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _basis(v, n):
    z = torch.zeros_like(n[:, 0])
    a = torch.stack([n[:, 2], z, -n[:, 0]], 1)
    b = torch.stack([z, n[:, 2], -n[:, 1]], 1)
    t = torch.where((n[:, 0].abs() > n[:, 1].abs())[:, None], a, b)
    b = torch.linalg.cross(n, t)
    t = torch.linalg.cross(b, n)
    return _unit(t * v[:, :1] + n * v[:, 1:2] + b * v[:, 2:])


def _box_image(seed, w, h, spp, depth, first):
    """Summed radiances (h, w, 3) of the Cornell box: every triangle tested, in 64 bits."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    spec = _spec("box", 1, seed)
    f64 = lambda x: torch.tensor(np.asarray(x, np.float32).astype(np.float64), device=dev)  # noqa: E731
    cam = spec["camera"]
    half = math.tan(math.radians(float(np.float32(cam["fov"]))) / 2)
    size = 2 * half / w
    eye = f64(cam["transform"]["translation"])
    bias = float(np.float32(1e-4))
    out = torch.zeros(w * h, 3, dtype=torch.float64, device=dev)
    pixel = torch.arange(w * h, device=dev, dtype=torch.int64)
    for p in range(first, first + spp):
        rng = _Pcg(torch.full_like(pixel, _wang(p)), pixel)
        x = -half + size * (pixel % w).double() + size * rng.uniform()
        y = half * h / w - size * torch.div(pixel, w, rounding_mode="floor").double() - size * rng.uniform()
        d = _unit(torch.stack([x, y, torch.ones_like(x)], 1))
        o = eye.expand_as(d)
        col = torch.ones_like(d)
        pid = pixel
        for _ in range(depth):
            t = torch.full_like(d[:, 0], math.inf)
            n = torch.zeros_like(d)
            mat = torch.full_like(pid, -1)
            for inst in spec["instances"]:
                m = _matrix(inst["transform"])
                inv = torch.tensor(np.linalg.inv(m), device=dev)
                oo, dd = o @ inv[:3, :3].T + inv[:3, 3], d @ inv[:3, :3].T
                mesh = spec["meshes"][inst["mesh"]]
                for tri in np.asarray(mesh["indices"]):
                    v0, v1, v2 = (f64(mesh["positions"][i]) for i in tri)
                    e1, e2 = v1 - v0, v2 - v0
                    P = torch.linalg.cross(dd, e2.expand_as(dd))
                    det = P @ e1
                    T = oo - v0
                    u = (T * P).sum(1) / det
                    Q = torch.linalg.cross(T, e1.expand_as(T))
                    v = (dd * Q).sum(1) / det
                    s = (Q @ e2) / det
                    hit = (det.abs() >= 2.0 ** -23) & (u >= 0) & (v >= 0) & (u + v <= 1) & (s > 0) & (s < t)
                    t = torch.where(hit, s, t)
                    ng = _unit((torch.linalg.cross(e1, e2) @ inv[:3, :3])[None])
                    n = torch.where(hit[:, None], ng, n)
                    mat = torch.where(hit, inst["material"], mat)
            alb = f64([x["albedo"] for x in spec["materials"]])[mat.clamp(min=0)] * (mat >= 0)[:, None]
            col = col * alb
            lit = mat == 3
            out[pid[lit]] += col[lit]
            n = torch.where(((n * d).sum(1) > 0)[:, None], -n, n)
            u1, u2 = rng.uniform(), rng.uniform()
            r, a = u1.sqrt(), 2 * math.pi * u2
            nd = _basis(torch.stack([r * a.cos(), (1 - u1).clamp(min=0).sqrt(), r * a.sin()], 1), n)
            on = (mat >= 0) & ~lit
            o = (o + d * torch.where(on, t, torch.zeros_like(t))[:, None] + n * bias)[on]
            d, col, pid = nd[on], col[on], pid[on]
            rng.s, rng.inc = rng.s[on], rng.inc[on]
            if not len(pid):
                break
    return out.reshape(h, w, 3).cpu().numpy()


def exact(case, seed):
    """Cornell box images in 64 bits. Other scenes have none: their closest hits and lobe choices
    over up to 722,000 triangles would take minutes by brute force."""
    rng = np.random.RandomState((seed + 7) & 0x7FFFFFFF)
    first = int(rng.randint(0, 1 << 16))
    images, any_box = [], False
    for k, w, h, spp, depth in _requests(case):
        box = k == "box" and w * h * spp <= 1 << 22
        any_box |= box
        images.append({"sum": _box_image(seed, w, h, spp, depth, first) if box else None, "pixels": None})
    return {"images": images} if any_box else None
