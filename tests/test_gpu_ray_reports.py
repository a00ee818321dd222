"""What ray queries report, formed on the device from the records' own ids: against the FP64 oracle's ids
on scenes that mix triangles, spheres, quads, shapes, lights and instances, for counts around a
workgroup, through the query kernel and the closest-hit stage; outputs the caller does not ask for."""
import ctypes as C

import numpy as np
import pytest

import oracle_py as O
from cortexraytracercuda_amd import Renderer, scenes, _abi as A

pytestmark = pytest.mark.gpu


def _mixed():
    s = scenes.shapes_scene()
    m = s.lambertian(None, (0.4, 0.5, 0.6))
    s.quad((-0.9, -0.9, -0.95), (0.4, 0.0, 0.0), (0.0, 0.5, 0.0), m)
    s.sphere((0.4, 0.5, -0.5), 0.2, m)
    s.sphere((-0.4, 0.4, -0.2), 0.1, m)
    return s


def _rays(n, seed, spread):
    rng = np.random.default_rng(seed)
    r = np.empty((n, 8), np.float32)
    r[:, 0:3] = rng.uniform(-spread, spread, (n, 3))
    r[:, 3] = 1e-5
    r[:, 4:7] = rng.normal(size=(n, 3))
    r[:, 7] = 3e38
    return r


@pytest.mark.parametrize("n", [1, 63, 256, 257, 5003])
def test_reported_ids(n):
    cases = [(_mixed(), 0.9), (scenes.instanced_scene(seed=2, n_instances=48, n_textures=2, tex_size=16, nu=12, nv=8, extent=8.0), 8.0)]
    with Renderer(max_paths=1 << 18) as r:
        for s, spread in cases:
            sid = r.upload(s)
            rays = _rays(n, 3, spread)
            prim, inst, t, uv = r.trace_rays(sid, rays)
            oprim, oinst, ot, _ = O.trace(s, rays.astype(np.float64), camera=False, precision=64, accel=1)
            # shape rims and instance ties may go the other way in FP32: at most one ray in a thousand
            same = prim == oprim
            assert (~same).sum() <= max(1, n // 1000)
            assert np.array_equal(inst[same], oinst[same])
            hit = same & (oprim >= 0)
            assert np.allclose(t[hit], ot[hit], rtol=1e-5, atol=1e-5)
            miss = prim < 0
            assert np.all(inst[miss] == -1) and np.all(t[miss] == 0) and np.all(uv[miss] == 0)
            sprim, sinst, st, _ = r.trace_rays(sid, rays, stage=True)
            assert sprim.shape == (n,) and np.all((sprim < 0) == (st == 0)) and np.all(sinst[sprim < 0] == -1)


def test_reports_only_what_is_asked_for():
    with Renderer(max_paths=1 << 18) as r:
        sid = r.upload(_mixed())
        rays = _rays(301, 5, 0.9)
        prim, inst, t, uv = r.trace_rays(sid, rays)
        only = np.zeros(301, np.float32)
        A.check(r.lib.crt_trace_rays(r.h, sid, rays.ctypes.data_as(C.POINTER(C.c_float)), 301, 0, None, None,
                                     only.ctypes.data_as(C.POINTER(C.c_float)), None))
        assert np.array_equal(only, t)
