"""Every value that a ray query reports: coordinates against the hit point, ids, instances, distances and
coordinates of the closest-hit stage against the query kernel's, and each output asked for alone."""
import ctypes as C

import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, scenes, _abi as A

pytestmark = pytest.mark.gpu


def _rays(n, seed, spread):
    rng = np.random.default_rng(seed)
    r = np.empty((n, 8), np.float32)
    r[:, 0:3] = rng.uniform(-spread, spread, (n, 3))
    r[:, 3] = 1e-5
    r[:, 4:7] = rng.normal(size=(n, 3))
    r[:, 7] = 3e38
    r[0, 0:3], r[0, 4:7] = (0.0, 0.0, 0.0), (0.01, -0.2, -0.45)   # onto the sphere in the middle
    return r


@pytest.mark.parametrize("n", [1, 64, 257, 4099])
def test_coordinates_give_the_hit_point(n):
    """v0 + u (v1 - v0) + v (v2 - v0) is o + t d. In 24 bits each side is off by some 16 roundings of a
    length of up to 3, over the cosine with the normal: 6e-5 from a cosine of 0.05 on. A swap of the
    coordinates, or another ray's, moves the point by about an edge, 0.02 and more."""
    s = scenes.sphere_mesh_scene(5000, seed=1)
    corners = np.concatenate([m["positions"].astype(np.float64)[m["indices"].reshape(-1, 3)] for m in s.meshes])
    first = len(s.lights) + len(s.spheres) + len(s.quads)   # triangles come behind the light, the spheres and the quads
    with Renderer(max_paths=1 << 18) as r:
        sid = r.upload(s)
        rays = _rays(n, 3, 0.9)
        prim, inst, t, uv = r.trace_rays(sid, rays)
    o, d = rays[:, 0:3].astype(np.float64), rays[:, 4:7].astype(np.float64)
    on_mesh = prim >= first
    assert on_mesh[0] and on_mesh.sum() >= n // 8
    tri = corners[prim[on_mesh] - first]
    normal = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    dm = d[on_mesh]
    cos = np.abs((normal * dm).sum(1)) / np.linalg.norm(normal, axis=1) / np.linalg.norm(dm, axis=1)
    u, v = uv[on_mesh, 0:1].astype(np.float64), uv[on_mesh, 1:2].astype(np.float64)
    at = tri[:, 0] + u * (tri[:, 1] - tri[:, 0]) + v * (tri[:, 2] - tri[:, 0])
    off = np.linalg.norm(at - (o[on_mesh] + t[on_mesh, None].astype(np.float64) * dm), axis=1)
    assert (off[cos >= 0.05] <= 1e-4).all()


SCENES = {
    "shapes": (scenes.shapes_scene, 0.9),
    "mesh": (lambda: scenes.sphere_mesh_scene(5000, seed=1), 0.9),
    "instanced": (lambda: scenes.instanced_scene(seed=2, n_instances=48, n_textures=2, tex_size=16, nu=12, nv=8, extent=8.0), 8.0),
}


@pytest.mark.parametrize("kind", sorted(SCENES))
@pytest.mark.parametrize("n", [1, 256, 5003])
def test_the_stage_reports_what_the_query_reports(kind, n):
    """Lights apart, whose back faces the stage's rays pass. Both answer each query exactly; distances and
    coordinates come from the same float expressions (1e-5 and 1e-4 allow for another order of them)."""
    make, spread = SCENES[kind]
    s = make()
    with Renderer(max_paths=1 << 18) as r:
        sid = r.upload(s)
        rays = _rays(n, 7, spread)
        prim, inst, t, uv = r.trace_rays(sid, rays)
        sprim, sinst, st, suv = r.trace_rays(sid, rays, stage=True)
    plain = prim >= len(s.lights) + len(s.sphere_lights)
    assert plain.any() or n == 1
    assert np.array_equal(sprim[plain], prim[plain]) and np.array_equal(sinst[plain], inst[plain])
    assert np.allclose(st[plain], t[plain], rtol=1e-5, atol=1e-6) and np.allclose(suv[plain], uv[plain], rtol=0, atol=1e-4)
    assert np.array_equal(sprim[prim < 0], prim[prim < 0])


def test_each_output_alone():
    f, i = C.POINTER(C.c_float), C.POINTER(C.c_int32)
    with Renderer(max_paths=1 << 18) as r:
        sid = r.upload(SCENES["instanced"][0]())
        rays = _rays(301, 5, 8.0)
        whole = r.trace_rays(sid, rays)
        for k, (like, kind) in enumerate(zip(whole, (i, i, f, f))):
            out = np.zeros_like(like)
            args = [None] * 4
            args[k] = out.ctypes.data_as(kind)
            A.check(r.lib.crt_trace_rays(r.h, sid, rays.ctypes.data_as(f), 301, 0, *args))
            assert np.array_equal(out, like), k
