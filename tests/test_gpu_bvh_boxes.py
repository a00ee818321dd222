"""GPU check of the device build's node boxes at the sizes where the range tree over the sorted
primitives has edges: its smallest sizes, one level of workgroups more or less, odd levels."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer
from cortexraytracercuda_amd.scene import Scene

pytestmark = pytest.mark.gpu


def _soup(n):
    g = np.random.default_rng(n)
    s = Scene()
    m = s.lambertian("grey", (0.7, 0.6, 0.5))
    v = (g.uniform(-1, 1, (n, 1, 3)) + g.normal(0, 0.5 * n ** -0.33, (n, 3, 3))).astype(np.float32)
    s.mesh(v.reshape(-1, 3), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), m)
    return s


@pytest.mark.parametrize("width", [4, 2])
@pytest.mark.parametrize("n", [2, 3, 5, 255, 256, 257, 511, 513, 65535, 65537, 70001])
def test_node_boxes_at_the_edges_of_the_range_tree(n, width):
    """Every node box holds its children (read back and verified), and closest hits equal the host tree's."""
    s = _soup(n)
    g = np.random.default_rng(1)
    one = np.ones((4096, 1))
    rays = np.concatenate([g.uniform(-1.5, 1.5, (4096, 3)), 1e-4 * one, g.normal(0, 1, (4096, 3)), 1e30 * one], 1)
    rays = rays.astype(np.float32)
    hits = {}
    for builder in ("host", "device"):
        with Renderer(bvh_builder=builder, bvh_width=width) as r:
            sid = r.upload(s)
            assert r.info(sid)["builder"] == builder
            r.verify(sid)
            hits[builder] = r.trace_rays(sid, rays)
    for a, b in zip(hits["host"], hits["device"]):
        assert np.array_equal(a, b, equal_nan=True)
