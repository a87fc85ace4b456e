"""The work a user of little_renderer_amd has it do, as cases that can be timed and compared.

Every case goes through the package's public entry points as a program calls them. The kinds:

  image      one picture of a resident scene (PtScene.render): a preview or a still
  jobs       many render jobs over one engine (Engine.submit / drain / image / release)
  frames     an instanced scene's frames: the moved instances' poses sent, the top level built
             again, the frame rendered under the sky
  caustics   one picture with light-traced caustics (PtScene.render_job, photons > 0)
  build      one BVH over boxes (Context.build), by either builder
  walk       a batch of rays against one binary BVH (Context.trace), closest or first hits
  rays       a batch of rays against a resident scene (lrh_pt_scene_trace), closest or first hits
  denoise    the variance-steered filter over a picture (Context.denoise)

Scenes, sizes and sample counts are the benchmark's and the tests' (a soup of 1k to 500k triangles
with 14 GGX materials, the Cornell room, the caustics room, 5001 instances; 256 x 256 to 1920 x
1080; 1 to 64 samples a pixel; up to 16M boxes), with ragged sizes beside them.
"""
import ctypes
import math

import numpy as np
import torch

import little_renderer_amd as lr

TMAX = 4.0           # rays end here, past every shape: a miss's t


def listed():
    return [
        # the smallest picture a program asks for: a one-sample preview of a room of 35 shapes
        # (launches and host round trips count)
        {"name": "preview_cornell", "kind": "image", "scene": "cornell", "tris": 0, "w": 256, "h": 256, "spp": 1},
        # a still of a mid-sized scene
        {"name": "still_soup", "kind": "image", "scene": "soup", "tris": 100000, "w": 1280, "h": 720, "spp": 8},
        # a render queue: 8 jobs on 8 scenes, sizes as the batched benchmark draws them
        {"name": "jobs_mixed", "kind": "jobs", "depth": 8, "mis": True,
         "jobs": "1200:1920x1080:4 500000:1280x720:16 8000:512x512:64 60000:1920x1080:1 250000:512x512:16 "
                 "3000:256x256:64 120000:1280x720:4 20000:256x256:1"},
        # a serving engine's light load: ten thumbnails of odd sizes
        {"name": "jobs_thumbnails", "kind": "jobs", "depth": 8, "mis": True,
         "jobs": "1000:160x120:4 5000:201x133:2 30000:256x256:1 1000:97x64:8 5000:320x180:1 30000:199x251:2 "
                 "1000:256x144:4 5000:128x128:4 30000:150x150:3 1000:75x211:1"},
        # two frames of a moving scene: 2000 of 5001 instances moved, a top level each, 1 sample
        {"name": "frames_instanced", "kind": "frames", "dynamic": 2000, "static": 3000, "props": 20, "hulls": 8, "sky": 2048,
         "w": 1280, "h": 720, "spp": 1},
        # glass and mirror balls under a lamp, a light path a pixel and pass
        {"name": "caustics", "kind": "caustics", "w": 512, "h": 512, "spp": 4, "photons": 1.0},
        # the builders: a large static scene's fast tree, a scene's good tree, a frame's top level
        {"name": "build_lbvh_4m", "kind": "build", "builder": "lbvh", "n": 4000000},
        {"name": "build_ploc_1m", "kind": "build", "builder": "ploc", "n": 1000000},
        {"name": "build_top_5001", "kind": "build", "builder": "ploc", "n": 5001},
        # the BVH-stress walk: a picture's primary rays through 1M triangles
        {"name": "walk_primary_1m", "kind": "walk", "builder": "ploc", "tris": 1000000, "w": 1920, "h": 1080, "aim": "camera",
         "any": False},
        # a batch of scene_intersect queries: rays from everywhere to everywhere
        {"name": "rays_scene", "kind": "rays", "builder": "ploc", "tris": 50000, "w": 600, "h": 500, "aim": "inside", "any": False},
        # a picture of few samples denoised
        {"name": "denoise_720p", "kind": "denoise", "w": 1280, "h": 720, "spp": 4, "passes": 5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["image", "jobs", "jobs", "frames", "caustics", "build", "build", "walk", "rays", "denoise"])
    if kind == "image":
        w = _log(rng, 64, 1920)
        h = max(33, int(w * rng.uniform(0.5, 1.0)))
        spp = max(1, min(64, _log(rng, 1, 64), 20000000 // (w * h)))
        scene = rng.choice(["cornell", "soup", "soup"])
        return {"kind": kind, "scene": scene, "tris": 0 if scene == "cornell" else _log(rng, 1000, 500000), "w": w, "h": h, "spp": spp}
    if kind == "jobs":
        specs, left = [], 40000000
        for _ in range(rng.randint(2, 10)):
            w = _log(rng, 64, 1920)
            h = max(33, int(w * rng.uniform(0.5, 1.0)))
            spp = max(1, min(rng.choice([1, 2, 4, 7, 16, 64]), left // (w * h)))
            if w * h * spp > left:
                break
            left -= w * h * spp
            specs.append("%d:%dx%d:%d" % (_log(rng, 1000, 300000), w, h, spp))
        return {"kind": kind, "depth": rng.choice([3, 5, 8, 8, 12]), "mis": rng.random() < 0.8, "jobs": " ".join(specs)}
    if kind == "frames":
        w = _log(rng, 200, 1600)
        return {"kind": kind, "dynamic": _log(rng, 20, 2000), "static": _log(rng, 20, 3000), "props": rng.randint(2, 20),
                "hulls": rng.randint(1, 8), "sky": rng.choice([512, 1000, 2048]), "w": w, "h": max(100, int(w * rng.uniform(0.5, 0.8))),
                "spp": rng.choice([1, 1, 2, 4])}
    if kind == "caustics":
        w = _log(rng, 64, 800)
        return {"kind": kind, "w": w, "h": max(50, int(w * rng.uniform(0.6, 1.0))), "spp": rng.randint(1, 16),
                "photons": rng.choice([0.25, 1.0, 2.0])}
    if kind == "build":
        builder = rng.choice(["lbvh", "ploc"])
        return {"kind": kind, "builder": builder, "n": _log(rng, 100, 16000000 if builder == "lbvh" else 4000000)}
    if kind in ("walk", "rays"):
        w = _log(rng, 64, 1920)
        return {"kind": kind, "builder": rng.choice(["lbvh", "ploc"]), "tris": _log(rng, 1000, 1000000), "w": w,
                "h": max(33, int(w * rng.uniform(0.4, 0.8))), "aim": rng.choice(["camera", "inside"]), "any": rng.random() < 0.4}
    w = _log(rng, 64, 3840)
    return {"kind": kind, "w": w, "h": max(33, int(w * rng.uniform(0.4, 0.8))), "spp": rng.choice([1, 2, 4, 16]),
            "passes": rng.choice([3, 5, 5])}


# ---- inputs -------------------------------------------------------------------------------------

def _specs(text):
    out = []
    for s in text.split():
        n, wh, spp = s.split(":")
        w, h = wh.split("x")
        out.append((int(n), int(w), int(h), int(spp)))
    return out


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _soup(n, seed):
    """triangles in the unit cube, edge lengths log-normal about the spacing of a full scene: (n, 12) on the GPU"""
    g = _gen(seed, 1)
    c = torch.rand((n, 3), generator=g, device="cuda")
    size = 0.4 * float(n) ** (-1.0 / 3.0)
    e = []
    for _ in range(2):
        d = torch.randn((n, 3), generator=g, device="cuda")
        d = d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)
        e.append(d * torch.exp(0.5 * torch.randn((n, 1), generator=g, device="cuda")) * size)
    t = torch.zeros((n, 12), device="cuda")
    t[:, 0:3], t[:, 4:7], t[:, 8:11] = c - (e[0] + e[1]) / 3.0, e[0], e[1]
    return t


def _boxes(n, seed):
    """boxes of a scene's shapes: clusters of objects in a room, (n, 8) on the GPU"""
    g = _gen(seed, 2)
    k = max(1, int(n ** 0.5) // 4)
    centre = torch.rand((k, 3), generator=g, device="cuda") * 10.0
    spread = torch.exp(torch.randn((k, 1), generator=g, device="cuda")) * 0.5
    at = torch.randint(0, k, (n,), generator=g, device="cuda")
    p = centre[at] + torch.randn((n, 3), generator=g, device="cuda") * spread[at]
    half = torch.exp(0.5 * torch.randn((n, 3), generator=g, device="cuda")) * (2.0 * float(n) ** (-1.0 / 3.0))
    b = torch.zeros((n, 8), device="cuda")
    b[:, 0:3], b[:, 4:7] = p - half, p + half
    return b


def _rays(case, seed):
    """camera: a pinhole's rays, row by row, towards the unit cube; inside: from points in and around it"""
    w, h = case["w"], case["h"]
    g = _gen(seed, 3)
    r = torch.empty((w * h, 8), device="cuda")
    if case["aim"] == "camera":
        eye = torch.randn(3, generator=g, device="cuda")
        eye = 0.5 + 1.8 * eye / eye.norm()
        z = eye - 0.5
        z = z / z.norm()
        up = torch.tensor([0.0, 1.0, 0.0], device="cuda") if abs(float(z[1])) < 0.9 else torch.tensor([1.0, 0.0, 0.0], device="cuda")
        x = torch.linalg.cross(up, z)
        x = x / x.norm()
        y = torch.linalg.cross(z, x)
        u = (torch.arange(w, device="cuda") + 0.5) / w - 0.5
        v = 0.5 - (torch.arange(h, device="cuda") + 0.5) / h
        d = (u[None, :, None] * (0.8 * w / h) * x + v[:, None, None] * 0.8 * y - z).reshape(-1, 3)
        o = eye.expand(w * h, 3)
    else:
        o = torch.rand((w * h, 3), generator=g, device="cuda") * 1.4 - 0.2
        d = torch.rand((w * h, 3), generator=g, device="cuda") - o
    r[:, 0:3], r[:, 3] = o, 1e-4
    r[:, 4:7], r[:, 7] = d / d.norm(dim=1, keepdim=True).clamp_min(1e-12), TMAX
    return r


def _picture(case, seed):
    """a picture's sums, moments and guide: the inside of a room with a ball and a lamp, its surfaces textured, each sample
    log-normal about the light there"""
    w, h, spp = case["w"], case["h"], case["spp"]
    g = _gen(seed, 4)
    rnd = torch.rand(8, generator=g, device="cuda").tolist()
    u = ((torch.arange(w, device="cuda") + 0.5) / w - 0.5) * (w / h)
    v = 0.5 - (torch.arange(h, device="cuda") + 0.5) / h
    d = torch.stack([u[None, :].expand(h, w), v[:, None].expand(h, w), torch.full((h, w), -0.9, device="cuda")], -1)
    d = d / d.norm(dim=-1, keepdim=True)
    o = torch.tensor([0.3 * (rnd[0] - 0.5), 0.3 * (rnd[1] - 0.5), 0.9], device="cuda")
    # the walls of [-1, 1]^3 from inside
    t = (torch.where(d > 0, 1.0, -1.0) - o) / torch.where(d.abs() < 1e-9, 1e-9, d)
    z, axis = t.min(-1)
    n = torch.zeros_like(d).scatter_(-1, axis[..., None], 1.0) * -torch.sign(d)
    # a ball
    c = torch.tensor([rnd[2] - 0.5, -0.5, -0.3 * rnd[3]], device="cuda")
    b = (d * (c - o)).sum(-1)
    disc = b * b - ((c - o) ** 2).sum() + 0.4 ** 2
    tb = b - disc.clamp_min(0).sqrt()
    ball = (disc > 0) & (tb > 0) & (tb < z)
    p = o + d * torch.where(ball, tb, z)[..., None]
    n = torch.where(ball[..., None], (p - c) / 0.4, n)
    z = torch.where(ball, tb, z)
    lamp = (~ball) & (axis == 1) & (d[..., 1] > 0) & (p[..., 0].abs() < 0.3) & (p[..., 2].abs() < 0.3)
    check = ((p * (3.0 + 4.0 * rnd[4])).floor().sum(-1).remainder(2.0))[..., None]
    alb = 0.15 + 0.7 * check * torch.tensor([rnd[5], rnd[6], rnd[7]], device="cuda") + 0.1 * (1 - check)
    light = (0.2 + 0.8 * (n * (torch.tensor([0.0, 1.0, 0.0], device="cuda") - p)).sum(-1).clamp_min(0.0)) / (0.3 + p[..., 1].sub(1).square())
    acc = torch.zeros((h, w, 4), device="cuda")
    mom = torch.zeros((h, w, 2), device="cuda")
    lum = torch.tensor([0.2126, 0.7152, 0.0722], device="cuda")
    for _ in range(spp):
        s = light[..., None] * torch.exp(0.9 * torch.randn((h, w, 1), generator=g, device="cuda") - 0.405) * torch.ones(3, device="cuda")
        s = torch.where(lamp[..., None], torch.full_like(s, 15.0), s * alb)
        l = (torch.where(lamp[..., None], s, s / alb.clamp_min(1e-3)) * lum).sum(-1)
        acc[..., :3] += s
        mom += torch.stack([l, l * l], -1)
    acc[..., 3] = spp
    gd = torch.empty((h, w, 8), device="cuda")
    gd[..., 0:3], gd[..., 3] = n, z
    gd[..., 4:7] = torch.where(lamp[..., None], torch.ones_like(alb), alb)
    gd[..., 7] = lamp.float()
    return acc, mom, gd


# ---- what a program has in hand -----------------------------------------------------------------

class _Case:
    """a context and what lives on it, closed with the state"""

    def __init__(self, **kw):
        self.ctx = lr.Context(0)
        # work of torch's that the library has to wait for goes on the context's own stream
        self.stream = torch.cuda.ExternalStream(self.ctx.stream)
        self.__dict__.update(kw)

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.ctx.close()
        except Exception:
            pass


def _scene(ctx, sc, builder=lr.PLOC):
    return lr.PtScene(ctx, sc["prims"], sc["tris"], sc["mats"], sc["light"], sc["eps"], sc["margin"], builder=builder)


def prepare(case, seed):
    kind = case["kind"]
    s = _Case(case=case)
    ctx = s.ctx
    if kind == "image":
        w, h = case["w"], case["h"]
        if case["scene"] == "cornell":
            sc = lr.cornell(w, h, seed)
            s.cam = sc["cam"]
        else:
            sc = lr.batch_scene(case["tris"], seed)
            s.cam = lr.batch_camera(seed + 1, w, h)
        s.scene, s.seed = _scene(ctx, sc), seed
        s.accum = torch.zeros((h, w, 4), device="cuda")
    elif kind == "jobs":
        specs = _specs(case["jobs"])
        s.scenes, s.jobs, s.out, made = [], [], [], {}
        for k, (n, w, h, spp) in enumerate(specs):
            if n not in made:
                made[n] = _scene(ctx, lr.batch_scene(n, seed + n))
                s.scenes.append(made[n])
            s.jobs.append(lr.make_job(made[n], lr.batch_camera(seed + k, w, h), w, h, spp, seed=seed + 7 * k,
                                      max_depth=case["depth"], mis=case["mis"]))
            s.out.append(torch.zeros((h, w, 4), device="cuda"))
        depth = max(x.info()[0] for x in s.scenes)
        image = sum((w * h * 24 + 255) // 256 * 256 for _, w, h, _ in specs) + (1 << 20)
        s.engine = lr.Engine(ctx, slots_log2=22, max_tree_depth=depth, image_bytes=image)
    elif kind == "frames":
        w, h = case["w"], case["h"]
        frames = [lr.instanced_workload(seed, f, case["dynamic"], case["static"], case["props"], case["hulls"]) for f in (0, 1, 2)]
        f0 = frames[0]
        s.scene = lr.PtScene.instanced(ctx, f0["mtris"], f0["mesh_first"], f0["mats"], f0["instances"])
        s.scene.set_sky(lr.sky(case["sky"], 35.0, 60.0, sun_le=(5e4, 4.6e4, 4e4)))
        s.moved = np.arange(1, 1 + case["dynamic"], dtype=np.int32)
        s.poses = [f["instances"][s.moved] for f in frames[1:]]
        cam = lr.camera_make((0.0, 14.0, -30.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0, w / h)
        s.jobs = [lr.make_job(s.scene, cam, w, h, case["spp"], seed=seed + k, max_depth=8) for k in range(2)]
        s.out = [torch.zeros((h, w, 4), device="cuda") for _ in range(2)]
        s.engine = lr.Engine(ctx, slots_log2=22, max_tree_depth=s.scene.info()[0] + 32, image_bytes=w * h * 24 + (1 << 20))
    elif kind == "caustics":
        w, h = case["w"], case["h"]
        sc = lr.caustic_scene(w, h, seed)
        s.scene = _scene(ctx, sc)
        s.job = lr.make_job(s.scene, sc["cam"], w, h, case["spp"], seed=seed, max_depth=8, photons=case["photons"])
        s.accum = torch.zeros((h, w, 4), device="cuda")
    elif kind == "build":
        n = case["n"]
        s.boxes = _boxes(n, seed)
        s.nodes = torch.zeros((2 * n - 1, 8), dtype=torch.int32, device="cuda")
        s.aux = torch.zeros(n, dtype=torch.int32, device="cuda")
    elif kind == "walk":
        n = case["tris"]
        s.tris, s.rays = _soup(n, seed), _rays(case, seed)
        boxes = torch.empty((n, 8), device="cuda")
        s.nodes = torch.zeros((2 * n - 1, 8), dtype=torch.int32, device="cuda")
        s.aux = torch.zeros(n, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        ctx.tri_boxes(s.tris, boxes)
        s.depth = ctx.build(boxes, n, s.nodes, s.aux, builder=lr.PLOC if case["builder"] == "ploc" else lr.LBVH).depth
        s.hits = torch.zeros((s.rays.shape[0], 4), device="cuda")
    elif kind == "rays":
        s.rays = _rays(case, seed)
        mats = (lr.Material * 1)()
        mats[0].albedo[:] = [0.5, 0.5, 0.5]
        sc = {"prims": None, "tris": _soup(case["tris"], seed).cpu().numpy(), "mats": mats, "light": -1, "eps": 1e-4, "margin": 1e-3}
        s.scene = _scene(ctx, sc, lr.PLOC if case["builder"] == "ploc" else lr.LBVH)
        s.hits = torch.zeros((s.rays.shape[0], 4), device="cuda")
    else:
        s.accum, s.moments, s.guide = _picture(case, seed)
        s.out = torch.zeros((case["h"], case["w"], 4), device="cuda")
    torch.cuda.synchronize()
    return s


# ---- one pass -------------------------------------------------------------------------------------

def _hits(s):
    words = s.hits.view(torch.int32)
    if s.case["any"]:   # which shape blocks a ray is the walk's own choice: whether one does is the answer
        with torch.cuda.stream(s.stream):
            return {"blocked": words[:, 1] != -1}
    return {"t": s.hits[:, 0], "id": words[:, 1], "b1": s.hits[:, 2], "b2": s.hits[:, 3]}


def run(s):
    case, ctx = s.case, s.ctx
    kind = case["kind"]
    if kind == "image":
        with torch.cuda.stream(s.stream):
            s.accum.zero_()
        s.scene.render(s.cam, case["w"], case["h"], case["spp"], s.accum, seed=s.seed)
        return s.accum
    if kind == "jobs":
        ids = [s.engine.submit(j) for j in s.jobs]
        s.engine.drain()
        for i, out in zip(ids, s.out):
            s.engine.image(i, out)
            s.engine.release(i)
        return s.out
    if kind == "frames":
        for poses, job, out in zip(s.poses, s.jobs, s.out):
            s.scene.move(s.moved, poses, builder=lr.PLOC)
            i = s.engine.submit(job)
            s.engine.drain()
            s.engine.image(i, out)
            s.engine.release(i)
        return s.out
    if kind == "caustics":
        with torch.cuda.stream(s.stream):
            s.accum.zero_()
        s.scene.render_job(s.job, s.accum)
        return s.accum
    if kind == "build":
        st = ctx.build(s.boxes, case["n"], s.nodes, s.aux, builder=lr.PLOC if case["builder"] == "ploc" else lr.LBVH)
        return {"nodes": s.nodes, "aux": s.aux, "depth": st.depth, "rounds": st.rounds, "clusters": st.clusters}
    if kind == "walk":
        ctx.trace(s.nodes, 0, s.aux, s.tris, s.rays, s.rays.shape[0], s.hits, s.depth, any_hit=case["any"])
        return _hits(s)
    if kind == "rays":
        p = ctypes.c_void_p
        rc = lr.lib().lrh_pt_scene_trace(ctx._c, s.scene._h, p(s.rays.data_ptr()), s.rays.shape[0], 1 if case["any"] else 0,
                                         p(s.hits.data_ptr()))
        if rc:
            raise lr.LrhError(lr.lib().lrh_last_error().decode())
        return _hits(s)
    ctx.denoise(s.accum, s.moments, s.guide, case["w"], case["h"], s.out, passes=case["passes"])
    return s.out


# ---- what a pass cannot do without -----------------------------------------------------------------

def work(case):
    """Bytes: inputs once, outputs once. Operations: a ray's boxes (about 72 slab tests of 14
    operations down a tree of this size) and 2 shapes of 45; 2.4 rays and 1.6 shaded vertices of 400
    a path; a filter tap's 60."""
    kind = case["kind"]
    ray, vertex = 72 * 14 + 2 * 45, 400
    path = 2.4 * ray + 1.6 * vertex
    if kind == "image":
        return {"bytes": 48 * case["tris"] + 32 * case["w"] * case["h"], "flops": path * case["w"] * case["h"] * case["spp"]}
    if kind == "jobs":
        specs = _specs(case["jobs"])
        return {"bytes": sum(48 * n + 16 * w * h for n, w, h, _ in specs), "flops": path * sum(w * h * spp for _, w, h, spp in specs)}
    if kind == "frames":
        ninst = 1 + case["dynamic"] + case["static"]
        return {"bytes": 2 * (56 * case["dynamic"] + 112 * ninst + 6 * case["sky"] ** 2 + 16 * case["w"] * case["h"]),
                "flops": 2 * path * 1.4 * case["w"] * case["h"] * case["spp"]}
    if kind == "caustics":
        n = case["w"] * case["h"] * case["spp"]
        return {"bytes": 32 * case["w"] * case["h"], "flops": (path + case["photons"] * (1.3 * ray + vertex)) * n}
    if kind == "build":
        return {"bytes": (32 + 64 + 4) * case["n"], "flops": 100 * case["n"]}
    if kind in ("walk", "rays"):
        n = case["w"] * case["h"]
        return {"bytes": 48 * n + (48 + 64 + 4) * case["tris"], "flops": ray * n}
    n = case["w"] * case["h"]
    return {"bytes": (16 + 8 + 32 + 16) * n, "flops": 25 * 60 * case["passes"] * n}


def tolerance(case):
    """Measured: the library compiled with fused multiply-adds against the library as it is (without),
    about four times what the outputs differed by. One hit at a shape's edge that becomes a miss, or
    one path that takes another turn at a random decision, is a whole pixel's difference."""
    kind = case["kind"]
    if kind == "build":
        return "exact"
    if kind in ("walk", "rays"):
        return {"rel": 1e-2, "max": 0.99, "differ": 1e-4}
    if kind == "denoise":
        return {"rel": 4e-5, "max": 5e-3}
    return {"rel": 6e-3, "max": 0.99}


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _exact_hits(case, seed):
    """every ray against every triangle, in 64 bits"""
    n, m = case["tris"], case["w"] * case["h"]
    if case["any"] or n * m > 2e10:
        return None
    tris, rays = _soup(n, seed).double(), _rays(case, seed).double()
    q, e1, e2 = tris[:, 0:3], tris[:, 4:7], tris[:, 8:11]
    T = torch.full((m,), TMAX, dtype=torch.float64, device="cuda")
    B1, B2 = torch.zeros_like(T), torch.zeros_like(T)
    # with o, d: det = d . (e2 x e1); each of the three numerators is linear in (o x d, d, o, 1)
    c = torch.linalg.cross(e2, e1)                                  # u . (d x v) = d . (v x u)
    step = max(1, int(4e7) // n)
    for a in range(0, m, step):
        o, d = rays[a:a + step, 0:3], rays[a:a + step, 4:7]
        od = torch.linalg.cross(o, d)
        det = d @ c.T
        inv = 1.0 / det
        # (o - q) . (d x v) = v . ((o - q) x d) = v . (o x d) - v . (q x d) = v . (o x d) + d . (q x v)
        b1 = (od @ e2.T + d @ torch.linalg.cross(q, e2).T) * inv
        # d . ((o - q) x u) = -u . ((o - q) x d)
        b2 = -(od @ e1.T + d @ torch.linalg.cross(q, e1).T) * inv
        # v . ((o - q) x u) = (o - q) . (u x v)
        t = (-(o @ c.T) + (q * c).sum(1)) * inv
        ok = (det.abs() >= 1e-12) & (b1 >= 0) & (b1 <= 1) & (b2 >= 0) & (b1 + b2 <= 1) & (t > rays[a:a + step, 3:4]) & (t < TMAX)
        t = torch.where(ok, t, TMAX)
        k = t.argmin(1, keepdim=True)
        hit = ok.gather(1, k)[:, 0]
        T[a:a + step] = t.gather(1, k)[:, 0]
        B1[a:a + step] = torch.where(hit, b1.gather(1, k)[:, 0], 0.0)
        B2[a:a + step] = torch.where(hit, b2.gather(1, k)[:, 0], 0.0)
    return {"t": T, "id": None, "b1": B1, "b2": B2}


def _hash32(x):
    m = 0xffffffff
    x = x ^ (x >> 16)
    x = (x * 0x7feb352d) & m
    x = x ^ (x >> 15)
    x = (x * 0x846ca68b) & m
    return x ^ (x >> 16)


def _exact_denoise(case, seed):
    """the filter on unpacked 64-bit numbers (the passes' 16-bit packing left out)"""
    acc, mom, gd = (x.double() for x in _picture(case, seed))
    h, w = case["h"], case["w"]
    n, z, alb, lamp = gd[..., 0:3], gd[..., 3], gd[..., 4:7], gd[..., 7] != 0
    wt = torch.tensor([0.2126, 0.7152, 0.0722], dtype=torch.float64, device="cuda")
    k = acc[..., 3:4].clamp_min(1.0)
    mean = acc[..., :3] / k
    irr = torch.where(lamp[..., None], mean, mean / alb.clamp_min(1e-3))
    Y, X = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
    if case["spp"] >= 4:
        el = mom[..., 0] / k[..., 0]
        var = (mom[..., 1] / k[..., 0] - el * el).clamp_min(0.0) / k[..., 0]
    else:
        s1, s2, cnt = (torch.zeros((h, w), dtype=torch.float64, device="cuda") for _ in range(3))
        lum = irr @ wt
        for dy in range(-3, 4):
            for dx in range(-3, 4):
                qy, qx = Y + dy, X + dx
                inside = (qy >= 0) & (qy < h) & (qx >= 0) & (qx < w)
                qy, qx = qy.clamp(0, h - 1), qx.clamp(0, w - 1)
                ok = (inside & (lamp[qy, qx] == lamp) & ((n[qy, qx] * n).sum(-1) >= 0.9)).double()
                l = lum[qy, qx]
                s1, s2, cnt = s1 + ok * l, s2 + ok * l * l, cnt + ok
        cnt = cnt.clamp_min(1.0)
        var = (s2 / cnt - (s1 / cnt) ** 2).clamp_min(0.0)
    var = torch.where(lamp, torch.zeros_like(var), var)
    hb = [1 / 16, 1 / 4, 3 / 8, 1 / 4, 1 / 16]
    zc = torch.where(lamp, torch.full_like(z, 2e38 - 1.0), z)
    out = irr
    for p in range(case["passes"]):
        step, last = 1 << p, p == case["passes"] - 1
        vb, vw = torch.zeros_like(var), 0.0
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                q = (0.25 if dx else 0.5) * (0.25 if dy else 0.5)
                vb, vw = vb + q * var[(Y + dy).clamp(0, h - 1), (X + dx).clamp(0, w - 1)], vw + q
        vb = vb / vw
        lp = out @ wt
        gx = torch.minimum((zc - zc[Y, (X - 1).clamp_min(0)]).abs(), (zc - zc[Y, (X + 1).clamp_max(w - 1)]).abs())
        gy = torch.minimum((zc - zc[(Y - 1).clamp_min(0), X]).abs(), (zc - zc[(Y + 1).clamp_max(h - 1), X]).abs())
        rs = _hash32((((Y * w + X) * 0x9e3779b9) & 0xffffffff) ^ ((step * 0x85ebca6b) & 0xffffffff))
        jit = step // 2
        jn = 2 * jit + 1
        total, vsum, wsum = torch.zeros_like(out), torch.zeros_like(var), torch.zeros_like(var)
        for j in range(5):
            for i in range(5):
                ox = torch.full_like(X, (i - 2) * step)
                oy = torch.full_like(Y, (j - 2) * step)
                centre = i == 2 and j == 2
                if jit > 0 and not centre:
                    rs = _hash32(rs)
                    ox = ox + (((rs & 0xffff) * jn) >> 16) - jit
                    oy = oy + (((rs >> 16) * jn) >> 16) - jit
                qy, qx = Y + oy, X + ox
                ok = (qy >= 0) & (qy < h) & (qx >= 0) & (qx < w)
                qy, qx = qy.clamp(0, h - 1), qx.clamp(0, w - 1)
                s, sv = out[qy, qx], var[qy, qx]
                q = torch.full_like(var, hb[i] * hb[j])
                same = (ox == 0) & (oy == 0)
                f = torch.exp(-(lp - s @ wt).abs() / (4.0 * torch.maximum(vb, sv).sqrt() + 1e-6))
                f = f * (n * n[qy, qx]).sum(-1).clamp_min(0.0) ** 128
                f = f * torch.exp(-(zc - zc[qy, qx]).abs() / (gx * ox.abs() + gy * oy.abs() + 1e-3 * zc + 1e-6))
                f = torch.where(lamp[qy, qx] == lamp, f, torch.zeros_like(f))
                q = torch.where(ok, torch.where(same, q, q * f), torch.zeros_like(q))
                total, vsum, wsum = total + q[..., None] * s, vsum + q * q * sv, wsum + q
        o = total / wsum[..., None]
        out, var = torch.where(lamp[..., None], out, o), torch.where(lamp, var, vsum / (wsum * wsum))
        if last:
            out = torch.where(lamp[..., None], out, out * alb)
    return torch.cat([out, torch.ones((h, w, 1), dtype=torch.float64, device="cuda")], -1)


def exact(case, seed):
    """Builds give whole numbers and boxes without rounding. A rendered picture has no such value:
    a path in other arithmetic takes other turns at its random decisions (and tracing the whole
    scenes without a tree takes minutes)."""
    if case["kind"] in ("walk", "rays"):
        return _exact_hits(case, seed)
    if case["kind"] == "denoise" and case["w"] * case["h"] <= 4000000:
        return _exact_denoise(case, seed)
    return None
