"""Calls that fail half way leave no queued work behind that names their buffers: those go back to a cache
that other streams take from. On the CPU (hip_standin)."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, _abi as A, scenes
from hip_standin import standin, standin_lib  # noqa: F401


@pytest.mark.parametrize("normals", [False, True])
def test_a_device_build_that_fails_leaves_nothing_queued(standin, normals):
    s = scenes.sphere_mesh_scene(3000, seed=1)
    s.sphere((0.1, 0.2, 0.3), 0.2, s.lambertian(None, (0.5, 0.5, 0.5)))
    if normals:
        m = s.meshes[0]
        m["normals"] = np.ones_like(m["positions"])
    with Renderer(max_paths=4096, pass_paths=4096, bvh_builder="device") as r:
        # one source buffer after the other: those before it come from the cache, all but the last one
        for n in range(5 + normals):
            r.lib.crt_debug_fail_alloc(r.h, min(n, 1))
            with pytest.raises(A.CrtError, match="injected"):
                r.upload(s)
            assert standin.standin_pending() == 0, n


@pytest.mark.parametrize("stage", [False, True])
@pytest.mark.parametrize("n", [3, 100001])   # rays that go through the pinned ring, and beyond it
def test_a_ray_query_that_fails_leaves_nothing_queued(standin, stage, n):
    rays = np.ones((n, 8), np.float32)
    with Renderer(max_paths=4096, pass_paths=4096) as r:
        sid = r.upload(scenes.box_scene())
        for k in range(2 if stage else 1):   # closest hits, report
            standin.standin_fail_launch(k)
            with pytest.raises(A.CrtError, match="launch failed"):
                r.trace_rays(sid, rays, stage=stage)
            assert standin.standin_pending() == 0, k
    with Renderer(max_paths=4096, pass_paths=4096) as r:
        sid = r.upload(scenes.box_scene())
        for k in range(7 if stage else 2):   # one buffer after the other, those before it from the cache
            r.lib.crt_debug_fail_alloc(r.h, min(k, 1))
            with pytest.raises(A.CrtError, match="injected"):
                r.trace_rays(sid, rays, stage=stage)
            assert standin.standin_pending() == 0, k


def _batch(sids, n):
    return [dict(sid=sids[k % len(sids)], width=40 + k, height=30, spp=4, max_depth=3, seed=k, rng=("pcg", "minstd")[k % 2])
            for k in range(n)]


def test_a_batch_that_fails_leaves_nothing_queued(standin):
    """A launch that is refused while others are queued on the second stream; a request whose buffers cannot
    be had while the ones before it have theirs started."""
    with Renderer(max_paths=1 << 14, pass_paths=1 << 14) as r:
        sids = [r.upload(s) for s in (scenes.box_scene(), scenes.shapes_scene())]
        for k in range(1, 5):
            standin.standin_fail_launch(k)
            with pytest.raises(A.CrtError, match="launch failed"):
                r.render_batch(_batch(sids, 6))
            assert standin.standin_pending() == 0, k
        for k in (1, 3, 7):
            r.lib.crt_debug_fail_alloc(r.h, k)
            with pytest.raises(A.CrtError, match="injected"):
                r.render_batch([dict(j, width=900 + 100 * k, height=600 + 100 * k) for j in _batch(sids, 9)])
            assert standin.standin_pending() == 0, k
        _, st = r.render_batch(_batch(sids, 6))
        assert st["paths"] == sum(j["width"] * j["height"] * 4 for j in _batch(sids, 6))
        standin.standin_fail_launch(0)
        with pytest.raises(A.CrtError, match="launch failed"):
            r.autotune(sids[0], 40, 30, 4, 3)
        assert standin.standin_pending() == 0
