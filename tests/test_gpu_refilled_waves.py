"""Refilled waves (long launches on scenes of many nodes: a wave shades the lanes that have their hit and
gives them the next ray while the others go on) against the staged pipeline (extend_kernel=1) on the same
requests: sums, images and counts are equal bit for bit."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


def _room(shapes):
    """19,570 or more nodes, an emitter whose back face paths pass, spheres and, with `shapes`, a disk."""
    s = scenes.sphere_mesh_scene(50000, seed=4)
    s.omni_light((0.55, 0.45, -0.3), 0.12, rgb=(1.0, 0.8, 0.6), intensity=6.0, invisible=False)
    s.spot_light((0.0, 0.0, 0.8), (0.2, -1.0, 0.1), 35.0, 4.0, 0.3, rgb=(0.6, 0.8, 1.0), intensity=20.0, invisible=False)
    if shapes:
        s.disk((0.0, 0.6, 0.0), 0.3, 0.1, s.metal("plate", (0.8, 0.7, 0.6), fuzz=0.1))
    return s


SCENES = {"room": lambda: _room(False), "shapes": lambda: _room(True), "open": lambda: scenes.large_scene(levels=6, n_spheres=200)}


def _equal(a, b):
    (rgb0, acc0, st0), (rgb1, acc1, st1) = a, b
    assert np.array_equal(acc0, acc1, equal_nan=True)
    assert np.array_equal(rgb0, rgb1)
    for key in ("rays", "paths", "retraces", "light_pdf_tests"):
        assert st0[key] == st1[key], key


# just under and over the paths that a launch needs (6,291,456); ragged tiles; a sample range; long paths
@pytest.mark.parametrize("w,h,spp,depth,first,count", [(2048, 1024, 4, 8, 0, 3), (2047, 1024, 4, 8, 0, 3), (1021, 771, 9, 8, 0, 0),
                                                       (1024, 1024, 16, 5, 5, 9), (700, 1000, 9, 40, 0, 0)])
@pytest.mark.parametrize("kind", sorted(SCENES))
def test_refilled_waves_equal_stages(kind, w, h, spp, depth, first, count):
    s = SCENES[kind]()
    print(kind, w, h, spp, depth, flush=True)
    with Renderer() as r, Renderer(extend_kernel=1) as staged:
        a, b = r.upload(s), staged.upload(s)
        assert r.info(a)["num_nodes"] >= 1 << 14
        got = [x.render(sid, w, h, spp, depth, seed=3, sample_begin=first, sample_count=count) for x, sid in ((r, a), (staged, b))]
        _equal(*got)
        if kind != "open" and depth == 8:
            assert got[0][2]["retraces"] > 0


def test_most_samples_and_short_queues_equal_stages():
    """As many samples a pixel as a request may have (refilled waves keep 16 bits of a sample's number), and
    slot pools from none for a queue to one queue of the shortest a wave."""
    s = _room(False)
    with Renderer(extend_kernel=1) as staged:
        b = staged.upload(s)
        ref = [staged.render(b, 10, 10, 65536, 4, seed=3), staged.render(b, 1024, 1024, 9, 6, seed=3)]
    with Renderer() as r:
        _equal(r.render(r.upload(s), 10, 10, 65536, 4, seed=3), ref[0])
    for paths in (1 << 12, 1 << 16, 1 << 20):
        with Renderer(max_paths=paths, pass_paths=1 << 24) as r:
            _equal(r.render(r.upload(s), 1024, 1024, 9, 6, seed=3), ref[1])
