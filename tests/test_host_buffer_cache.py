"""The cache of released buffers gives way to what a call needs. On the CPU (hip_standin)."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, _abi as A, scenes
from hip_standin import standin, standin_lib  # noqa: F401


def test_the_cache_gives_way_when_device_memory_runs_out(standin):
    """A scene, a render and a query that fit once the buffers of earlier calls are given up."""
    box, mesh = scenes.box_scene(), scenes.sphere_mesh_scene(60000, seed=2)
    rays = np.ones((200000, 8), np.float32)
    with Renderer(max_paths=4096, pass_paths=4096) as r:
        sid = r.upload(box)
        before = standin.standin_allocated()
        r.trace_rays(sid, rays)
        cached = standin.standin_allocated() - before
        assert cached >= rays.shape[0] * 52
        for call in (lambda: r.upload(mesh), lambda: r.render(sid, 700, 700, 1, 2), lambda: r.trace_rays(sid, rays[:50000], stage=True)):
            # nothing free but what the cache holds
            standin.standin_memory_limit(standin.standin_allocated())
            call()
            standin.standin_memory_limit(0)
            r.trace_rays(sid, rays)
        standin.standin_memory_limit(standin.standin_allocated())
        with pytest.raises(A.CrtError, match="hipMalloc"):
            r.render(sid, 4096, 4096, 1, 2)


def test_the_cache_stays_within_the_budget(standin):
    """What a context holds in device memory does not exceed its budget between calls, whichever call filled
    the cache and whichever needs the room, and repeated calls keep their buffers."""
    n = 1 << 18
    rays = np.ones((n, 8), np.float32)
    mesh = scenes.sphere_mesh_scene(60000, seed=2)
    start = standin.standin_allocated()
    with Renderer(max_paths=4096, pass_paths=4096) as r:
        sid = r.upload(mesh)
        scene_bytes = r.info(sid)["device_bytes"]
        r.wait(r.submit(sid, 8, 8, 1, 2), 8, 8)
        reserved = r.memory()["reserved"]
    assert standin.standin_allocated() == start
    # a stage query takes 20 + 16 + 4 + 16 + 16 + 8 bytes a ray; the budget has room for 8 MB beside the scene
    assert n * 80 > scene_bytes + (8 << 20) + (4 << 20)
    with Renderer(max_paths=4096, pass_paths=4096, hbm_budget=reserved + scene_bytes + (8 << 20)) as r:

        def inside():   # size classes round a buffer up: 8 for 5.25 MB, 4 for 3
            return standin.standin_allocated() - start <= r.memory()["budget"] + (4 << 20)

        small = r.upload(scenes.box_scene())
        r.wait(r.submit(small, 8, 8, 1, 2), 8, 8)
        r.trace_rays(small, rays, stage=True)
        assert inside()
        sid = r.upload(mesh)
        assert inside()
        r.trace_rays(sid, rays, stage=True)
        assert inside()
        r.render(sid, 400, 400, 1, 2)
        assert inside()
        held = standin.standin_allocated()
        r.render(sid, 400, 400, 1, 2)
        assert standin.standin_allocated() == held
        for w in (400, 500, 8):
            r.wait(r.submit(sid, w, w, 1, 2), w, w)
            assert inside()
