"""The work that users of the renderer have it do, as a list of cases that can be timed.

A case is a dict of plain values. `prepare` makes what a program holds before the call (resident
scenes, rays, a render seed), `run` makes one call through the public Python interface and returns its
outputs (images, accumulation buffers, ray counts, hits), `work` says what the call cannot do without,
and `exact` gives closest hits in 64 bits by testing every primitive. `draw` gives more cases of the
ranges that the listed ones stand for.

Kinds of cases:
  render  one blocking render of a resident scene (Renderer.render)
  batch   several requests on several scenes in one call (Renderer.render_batch)
  serve   the same through the request queue (Renderer.submit, Renderer.wait)
  rays    closest hits of the caller's own rays (Renderer.trace_rays)
  build   a scene that arrives with its request: upload with the tree built on the GPU, the first
          image, release
Scenes are those of cortexraytracercuda_amd.scenes and a scene file; per seed their spheres,
instances and displacements differ.
"""
import copy
import functools
import math
import os

import numpy as np
import torch

from cortexraytracercuda_amd import Renderer, SceneFile, scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCENE_FILE = os.path.join(ROOT, "tests", "golden", "scenes", "shipped_all_lights_types.scene")


def listed():
    return [
        # a thumbnail of the small box scene, as an editor's preview shows it: launches and latency
        dict(name="box_64", kind="render", scene="box", detail=0, width=64, height=64, spp=16, depth=8, first=0, count=0,
             rng="pcg"),
        # the small box scene at the size that its workload is defined with
        dict(name="box_256", kind="render", scene="box", detail=0, width=256, height=256, spp=16, depth=8, first=0, count=0,
             rng="pcg"),
        # a mesh in the lit box at an odd size (no 8x8 tiling), a sample count that is not a square, few bounces
        dict(name="mesh_301x173", kind="render", scene="mesh", detail=30000, width=301, height=173, spp=10, depth=5, first=0,
             count=0, rng="pcg"),
        # a scene file with the image size, sample count and depth that it asks for, on the reference's own
        # random stream: the reference program's command line
        dict(name="file_512x388_minstd", kind="render", scene="file", detail=0, width=512, height=388, spp=50, depth=100,
             first=0, count=0, rng="minstd"),
        # disks, cylinders, a cone, checker and image textures, glass and metal at a video size
        dict(name="shapes_640x360", kind="render", scene="shapes", detail=0, width=640, height=360, spp=16, depth=8, first=0,
             count=0, rng="pcg"),
        # a closed diffuse room around a mesh of 2,000,000 triangles: incoherent bounces in a large tree
        dict(name="room_2m_1024", kind="render", scene="mesh", detail=2000000, width=1024, height=1024, spp=64, depth=8,
             first=0, count=0, rng="pcg"),
        # the benchmark's frame: 1,310,720 triangles and 500 spheres under a sky
        dict(name="large_1080p", kind="render", scene="large", detail=8, width=1920, height=1080, spp=64, depth=10, first=0,
             count=0, rng="pcg"),
        # one pass of a progressive render of 4,096 textured instances: one sample for each pixel of a 4K image
        dict(name="instanced_4k_pass", kind="render", scene="instanced", detail=4096, width=3840, height=2160, spp=16,
             depth=12, first=5, count=1, rng="pcg"),
        # a batch of uneven requests on six scenes
        dict(name="batch_12", kind="batch", scene="mesh", detail=500000, scenes=6, requests=12, width=1024, spp=64, depth=8,
             mix=4),
        # requests that wait in the service's queue at once, small ones among larger ones
        dict(name="serve_20", kind="serve", scene="mesh", detail=200000, scenes=4, requests=20, width=1024, spp=64, depth=8,
             mix=11),
        # closest hits of the caller's rays (visibility and picking): host arrays in, host arrays out
        dict(name="rays_200k", kind="rays", scene="large", detail=4, rays=200001),
        # a scene that was not seen before, at the service's door: tree built on the GPU, first image
        dict(name="build_300k", kind="build", scene="mesh", detail=300000, width=256, height=256, spp=4, depth=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_render(rng):
    scene = rng.choice(["box", "mesh", "mesh", "file", "shapes", "large", "instanced"])
    detail = {"box": lambda: 0, "file": lambda: 0, "shapes": lambda: 0, "mesh": lambda: _log_int(rng, 1e4, 2e6),
              "large": lambda: rng.randint(4, 8), "instanced": lambda: _log_int(rng, 64, 4096)}[scene]()
    stream = rng.choice(["pcg", "pcg", "pcg", "minstd"])
    # paths of one call: up to the listed cases' own (fewer on the stream that runs a pixel's samples in turn)
    most = 3e6 if stream == "minstd" else {"large": 1e8, "instanced": 8e6}.get(scene, 4e7)
    while True:
        width = _log_int(rng, 48, 2048)
        height = max(32, int(width * rng.choice([1.0, 0.75, 0.5625, 0.5625, rng.uniform(0.4, 1.3)])))
        spp = _log_int(rng, 1, 64)
        if width * height * spp <= most:
            break
    first, count = 0, 0
    if stream == "pcg" and spp >= 9 and rng.random() < 0.25:   # a sample range of a progressive render
        total = int(math.sqrt(spp)) ** 2
        first = rng.randrange(total)
        count = rng.randint(1, total - first)
    return dict(kind="render", scene=scene, detail=detail, width=width, height=height, spp=spp,
                depth=rng.choice([2, 4, 5, 8, 8, 10, 12]), first=first, count=count, rng=stream)


def draw(rng):
    kind = rng.choice(["render"] * 6 + ["batch", "serve", "rays", "build"])
    if kind == "render":
        return _draw_render(rng)
    if kind in ("batch", "serve"):
        return dict(kind=kind, scene="mesh", detail=_log_int(rng, 2e4, 4e5), scenes=rng.randint(2, 5),
                    requests=rng.randint(4, 12 if kind == "batch" else 20), width=_log_int(rng, 192, 1024),
                    spp=_log_int(rng, 4, 64), depth=rng.choice([4, 5, 8, 8]), mix=rng.randrange(1000))
    if kind == "rays":
        return dict(kind="rays", scene="large", detail=rng.randint(2, 7), rays=_log_int(rng, 1000, 1000000))
    return dict(kind="build", scene="mesh", detail=_log_int(rng, 1e4, 1e6), width=_log_int(rng, 64, 512),
                height=_log_int(rng, 64, 512), spp=_log_int(rng, 1, 9), depth=rng.choice([4, 8]))


# ------------------------------------------------------------------ scenes
@functools.lru_cache(maxsize=None)
def _renderer(builder):
    """The program's one renderer (two where it also serves scenes built on the GPU)."""
    return Renderer(bvh_builder=builder)


@functools.lru_cache(maxsize=2)
def _large_base(levels):
    return scenes.large_scene(seed=1, levels=levels, n_spheres=0)


@functools.lru_cache(maxsize=1)
def _instanced_base():
    return scenes.instanced_scene(seed=1, n_instances=0, n_textures=4, tex_size=2048, nu=50, nv=50)


def _copy(base):
    s = copy.copy(base)
    s.materials, s.spheres, s.instances = list(base.materials), list(base.spheres), list(base.instances)
    s.material_names = dict(base.material_names)
    return s


def _scene(name, detail, seed, aspect):
    """A scene of the named kind. The meshes and textures that do not depend on the seed are loaded once,
    as a program's assets are; spheres, instances and displacements come from the seed."""
    rng = np.random.default_rng([seed, 77])
    if name == "file":
        return SceneFile(SCENE_FILE)
    if name == "mesh":
        return scenes.sphere_mesh_scene(detail, seed=seed % 100000, aspect=aspect)
    if name == "large":
        s = _copy(_large_base(detail))
        s.set_camera((0.0, 4.0, 24.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), vfov=45.0, aspect_ratio=aspect, focus_dist=10.0)
        for _ in range(500):
            c, r, u = rng.uniform(-10.0, 10.0, 3), rng.uniform(0.1, 0.5), rng.random()
            if u < 0.6:
                m = s.lambertian(None, tuple(rng.uniform(0.1, 0.9, 3)))
            elif u < 0.9:
                m = s.metal(None, tuple(rng.uniform(0.1, 0.9, 3)), fuzz=float(rng.uniform(0.0, 0.5)))
            else:
                m = s.dielectric(None, 1.5)
            s.sphere(tuple(c), float(r), m)
        return s
    if name == "instanced":
        s = _copy(_instanced_base())
        s.set_camera((0.0, 10.0, 120.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), vfov=60.0, aspect_ratio=aspect, focus_dist=10.0)
        for k in range(detail):
            place = np.concatenate([scenes.random_rotation(rng) * rng.uniform(1.0, 2.5), rng.uniform(-50.0, 50.0, 3)[:, None]], 1)
            s.instance(0, place, material_override=s.material_names["tor%d" % (k % 4)])
        return s
    s = scenes.box_scene() if name == "box" else scenes.shapes_scene()
    s.set_camera((0.0, 0.0, 0.9), (0.0, 0.0, -1.0), (0.0, 1.0, 0.0), vfov=70.0, aspect_ratio=aspect, focus_dist=10.0)
    return s


class _Resident:
    """Scenes that a program keeps uploaded; given back with the object."""

    def __init__(self, renderer, descriptions):
        self.renderer = renderer
        self.ids = [renderer.upload(d) for d in descriptions]

    def __del__(self):
        for sid in self.ids:
            self.renderer.release(sid)


# ------------------------------------------------------------------ cases
def _requests(case, seed):
    """The requests of a batch or a queue: sizes by the case's mix, seeds by the seed."""
    rng = np.random.default_rng(case["mix"])
    sizes = [max(64, int(case["width"] * f)) for f in (0.25, 0.375, 0.5, 0.75, 1.0)]
    got = []
    for k in range(case["requests"]):
        side = int(rng.choice(sizes))
        got.append(dict(scene=k % case["scenes"], width=side, height=side, spp=int(rng.integers(1, case["spp"] + 1)),
                        max_depth=case["depth"], seed=1000 * (seed % 1000000) + k))
    return got


def _triangles(case):
    """Triangle counts of the scenes of a batch or a queue: spread over a factor of fifty."""
    n = case["scenes"]
    return [max(64, int(case["detail"] * 50.0 ** (-k / max(1, n - 1)))) for k in range(n)]


def _rays(case, seed):
    """Rays through the scene from points around it: origin, tmin, direction, tmax."""
    rng = np.random.default_rng([seed, 5])
    n = case["rays"]
    o = rng.uniform(-12.0, 12.0, (n, 3))
    d = rng.normal(size=(n, 3))
    d[::2] = rng.uniform(-3.5, 3.5, (n, 3))[::2] - o[::2]   # every second one towards the middle
    r = np.empty((n, 8), np.float32)
    r[:, 0:3], r[:, 3], r[:, 4:7], r[:, 7] = o, 1e-5, d, 3.0e38
    return r


def prepare(case, seed):
    kind = case["kind"]
    if kind == "build":
        return dict(kind=kind, case=case, seed=seed, renderer=_renderer("device"),
                    scene=_scene(case["scene"], case["detail"], seed, case["width"] / case["height"]))
    r = _renderer("host")
    if kind == "render":
        scene = _scene(case["scene"], case["detail"], seed, case["width"] / case["height"])
        return dict(kind=kind, case=case, seed=seed, renderer=r, held=_Resident(r, [scene]))
    if kind in ("batch", "serve"):
        held = _Resident(r, [_scene(case["scene"], t, seed + k, 1.0) for k, t in enumerate(_triangles(case))])
        jobs = [dict(q, sid=held.ids[q["scene"]]) for q in _requests(case, seed)]
        return dict(kind=kind, case=case, renderer=r, held=held, jobs=jobs)
    scene = _scene(case["scene"], case["detail"], seed, 16.0 / 9.0)
    return dict(kind=kind, case=case, renderer=r, held=_Resident(r, [scene]), rays=_rays(case, seed))


def run(state):
    r, c, kind = state["renderer"], state["case"], state["kind"]
    if kind == "render":
        rgb, accum, st = r.render(state["held"].ids[0], c["width"], c["height"], c["spp"], c["depth"], seed=state["seed"],
                                  rng=c["rng"], sample_begin=c["first"], sample_count=c["count"])
        return dict(rgb=rgb, accum=accum, rays=st["rays"], paths=st["paths"])
    if kind == "batch":
        images, st = r.render_batch(state["jobs"])
        return dict(rgb=[i[0] for i in images], accum=[i[1] for i in images], rays=st["rays"], paths=st["paths"])
    if kind == "serve":
        ids = [r.submit(q["sid"], q["width"], q["height"], q["spp"], q["max_depth"], seed=q["seed"], image_only=True)
               for q in state["jobs"]]
        done = [r.wait(i, q["width"], q["height"], want_accum=False) for i, q in zip(ids, state["jobs"])]
        return dict(rgb=[d[0] for d in done], rays=[d[2]["rays"] for d in done])
    if kind == "rays":
        prim, inst, t, uv = r.trace_rays(state["held"].ids[0], state["rays"])
        return dict(prim=prim, inst=inst, t=t, uv=uv)
    sid = r.upload(state["scene"])
    rgb, accum, st = r.render(sid, c["width"], c["height"], c["spp"], c["depth"], seed=state["seed"])
    r.release(sid)
    return dict(rgb=rgb, accum=accum, rays=st["rays"])


# ------------------------------------------------------------------ what a call cannot do without
# Floating operations: one four-wide box test is 4 * 12 multiply-adds and comparisons, one primitive test
# about 60, shading with its random draws about 150. Rays of a path on average, by scene: a closed
# room keeps a path alive to its depth, an open one lets most of them go.
_RAYS_PER_PATH = {"box": 4.0, "mesh": 4.0, "shapes": 4.0, "file": 1.5, "large": 1.45, "instanced": 1.6}


def _triangle_count(scene, detail):
    return {"mesh": lambda: detail + 12, "large": lambda: 20 * 4 ** detail, "instanced": lambda: 5000 * max(1, detail)}.get(
        scene, lambda: 12)()


def _scene_bytes(scene, detail):
    """Vertices and indices once (instances share their mesh and bring 64 bytes each)."""
    if scene == "instanced":
        return 5000 * 18 + 64 * detail + 4 * 2048 * 2048 * 4
    return _triangle_count(scene, detail) * 18 + 500 * 32


def _ray_flops(scene, detail):
    return 96.0 * max(1.0, math.log(_triangle_count(scene, detail) + 1, 4)) + 60.0


def _render_work(scene, detail, width, height, samples, depth):
    paths = float(width * height * samples)
    rays = paths * min(float(depth), _RAYS_PER_PATH[scene])
    return width * height * 19.0, rays * (_ray_flops(scene, detail) + 150.0)


def _samples(case):
    total = int(math.sqrt(case["spp"])) ** 2
    return min(total - case.get("first", 0), case.get("count", 0) or total)


def work(case):
    kind = case["kind"]
    if kind in ("render", "build"):
        out, flops = _render_work(case["scene"], case["detail"], case["width"], case["height"], _samples(case), case["depth"])
        return dict(bytes=out + _scene_bytes(case["scene"], case["detail"]), flops=flops)
    if kind in ("batch", "serve"):
        triangles = _triangles(case)
        moved, flops = float(sum(_scene_bytes("mesh", t) for t in triangles)), 0.0
        for q in _requests(case, 0):
            b, f = _render_work("mesh", triangles[q["scene"]], q["width"], q["height"], int(math.sqrt(q["spp"])) ** 2, case["depth"])
            moved, flops = moved + (b if kind == "batch" else b * 3.0 / 19.0), flops + f
        return dict(bytes=moved, flops=flops)
    return dict(bytes=case["rays"] * (32.0 + 20.0) + _scene_bytes(case["scene"], case["detail"]),
                flops=case["rays"] * _ray_flops(case["scene"], case["detail"]))


# ------------------------------------------------------------------ closest hits in 64 bits
def _exact_hits(scene, rays, device):
    """Distance and (u, v) of each ray's closest hit: every triangle, sphere and area light is tested in
    64 bits. Of hits whose distances are within 2^-20 of the nearest the lowest primitive counts, as
    the renderer defines it (lights, then spheres, then triangles)."""
    f64 = dict(dtype=torch.float64, device=device)
    ray = torch.as_tensor(rays.astype(np.float64), **f64)
    light, mesh = scene.lights[0], scene.meshes[0]
    pos = torch.as_tensor(mesh["positions"].astype(np.float64), **f64)
    tri = pos[torch.as_tensor(mesh["indices"].astype(np.int64), device=device)]
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    f32 = lambda v: torch.as_tensor(np.asarray(v, np.float32).astype(np.float64), **f64)  # noqa: E731
    sc, sr = f32([s["center"] for s in scene.spheres]), f32([s["radius"] for s in scene.spheres])
    q, lu, lv = f32(light["center"]), f32(light["u"]), f32(light["v"])
    n = torch.linalg.cross(lu, lv)
    inf = float("inf")
    ts, uvs = [], []
    step = max(1, 16_000_000 // max(1, tri.shape[0] + sc.shape[0]))
    for k in range(0, ray.shape[0], step):
        o, tmin, d = ray[k:k + step, 0:3], ray[k:k + step, 3:4], ray[k:k + step, 4:7]
        # area light: centre +- half an edge
        tl = ((q - o) @ n) / (d @ n)
        h = o + tl[:, None] * d - q
        lalpha, lbeta = (torch.linalg.cross(h, lv.expand_as(h)) @ n) / (n @ n), (torch.linalg.cross(lu.expand_as(h), h) @ n) / (n @ n)
        tl = torch.where((tl >= tmin[:, 0]) & (lalpha.abs() <= 0.5) & (lbeta.abs() <= 0.5), tl, torch.full_like(tl, inf))
        # spheres: the nearest root beyond tmin
        oc = o[:, None] - sc
        aa, hb = (d * d).sum(1, keepdim=True), (oc * d[:, None]).sum(2)
        disc = hb * hb - aa * ((oc * oc).sum(2) - sr * sr)
        root = disc.clamp(min=0).sqrt()
        t0, t1 = (-hb - root) / aa, (-hb + root) / aa
        tsph = torch.where(t0 > tmin, t0, torch.where(t1 > tmin, t1, torch.full_like(t0, inf)))
        tsph = torch.where(disc >= 0, tsph, torch.full_like(t0, inf))
        # triangles: the barycentric volumes as products of (d, o x d) with each edge's direction and moment
        m = torch.linalg.cross(o, d)
        n2 = torch.linalg.cross(e1, e2)
        det = d @ n2.T
        u = (d @ torch.linalg.cross(e2, a).T - m @ e2.T) / det
        v = (m @ e1.T - d @ torch.linalg.cross(e1, a).T) / det
        tt = ((a * n2).sum(1) - o @ n2.T) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (tt >= tmin)
        tt = torch.where(ok, tt, torch.full_like(tt, inf))
        every = torch.cat([tl[:, None], tsph, tt], 1)
        best = every.min(1).values
        first = (every <= best[:, None] * (1 + 2.0 ** -20)).to(torch.int8).argmax(1)
        t = every.gather(1, first[:, None])[:, 0]
        j = (first - 1 - sc.shape[0]).clamp(min=0)[:, None]
        uv = torch.stack([u.gather(1, j)[:, 0], v.gather(1, j)[:, 0]], 1)
        uv[(first >= 1) & (first <= sc.shape[0])] = 0.0
        uv = torch.where((first == 0)[:, None], torch.stack([lalpha + 0.5, lbeta + 0.5], 1), uv)
        miss = torch.isinf(t)
        t, uv = torch.where(miss, torch.zeros_like(t), t), torch.where(miss[:, None], torch.zeros_like(uv), uv)
        ts.append(t)
        uvs.append(uv)
    return torch.cat(ts).cpu().numpy(), torch.cat(uvs).cpu().numpy()


def exact(case, seed):
    """Closest hits have a value in 64 bits. An image is a sum over random paths, whose every float
    decision belongs to it: it has none but the same sums again."""
    if case["kind"] != "rays" or case["rays"] * (_triangle_count(case["scene"], case["detail"]) + 500) > 2e10:
        return None
    scene = _scene(case["scene"], case["detail"], seed, 16.0 / 9.0)
    t, uv = _exact_hits(scene, _rays(case, seed), "cuda" if torch.cuda.is_available() else "cpu")
    return dict(prim=None, inst=None, t=t, uv=uv)
