"""Results on their way to the caller's memory: image and accumulation buffer together below and above
one pinned chunk (1 MiB), above the size from which threads help (8 MiB) and above the whole ring
(32 MiB), with row counts that leave ragged last chunks. The image is the tonemap of the accumulation
buffer, value by value, and both equal the same render's served result."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


def _tonemap(acc, spp):
    x = np.nan_to_num(acc[..., :3], nan=0.0) * (np.float32(1.0) / np.float32(spp))
    x = np.clip(np.sqrt(x.astype(np.float32)), np.float32(0.0), np.float32(0.999))
    return (np.float32(255.99) * x).astype(np.uint8)


@pytest.mark.parametrize("width,height", [(1, 1), (61, 53), (233, 231), (256, 256), (640, 701), (1531, 1027), (2048, 1100)])
def test_images_and_sums_of_every_size_arrive_whole(width, height):
    s = scenes.box_scene()
    with Renderer(max_paths=1 << 22) as r:
        sid = r.upload(s)
        rgb, acc, st = r.render(sid, width, height, 1, 2, seed=5)
        assert np.all(acc[..., 3] == 1.0) and st["paths"] == width * height
        assert np.array_equal(rgb, _tonemap(acc, 1))
        only, none, _ = r.render(sid, width, height, 1, 2, seed=5, want_accum=False)
        assert none is None and np.array_equal(only, rgb)
        srgb, sacc, _ = r.wait(r.submit(sid, width, height, 1, 2, seed=5), width, height)
        assert np.array_equal(srgb, rgb) and np.array_equal(sacc, acc)


def test_a_batch_of_many_outputs_arrives_whole():
    """Small and large outputs in one list: pieces of different requests share the ring."""
    sizes = [(8, 8), (700, 640), (33, 7), (1024, 512), (5, 1), (640, 480), (512, 512)]
    with Renderer(max_paths=1 << 22) as r:
        sid = r.upload(scenes.box_scene())
        jobs = [dict(sid=sid, width=w, height=h, spp=1, max_depth=2, seed=k) for k, (w, h) in enumerate(sizes)]
        for j, (rgb, acc) in zip(jobs, r.render_batch(jobs)[0]):
            rgb1, acc1, _ = r.render(sid, j["width"], j["height"], 1, 2, seed=j["seed"])
            assert np.array_equal(acc, acc1) and np.array_equal(rgb, rgb1)
