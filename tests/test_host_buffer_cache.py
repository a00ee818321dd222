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
