"""Whole-path launches (one launch follows the paths of a request to their end) against the staged
pipeline (extend_kernel=1) on the same requests: the same float operations per path and the same sums
per pixel, so accumulation buffers, images and every count are equal bit for bit."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


def _lit():
    """An omni light and a visible spot light around the camera: camera rays pass its back face and carry
    its white on."""
    s = scenes.box_scene()
    s.omni_light((0.55, 0.45, -0.3), 0.12, rgb=(1.0, 0.8, 0.6), intensity=6.0, invisible=False)
    s.spot_light((0.0, 0.0, 0.8), (0.2, -1.0, 0.1), 35.0, 4.0, 0.3, rgb=(0.6, 0.8, 1.0), intensity=20.0, invisible=False)
    return s


def _instanced(shapes):
    s = scenes.instanced_scene(seed=2, n_instances=40, n_textures=2, tex_size=32, nu=12, nv=8, extent=10.0)
    if shapes:
        m = s.metal("tube", (0.8, 0.7, 0.6), fuzz=0.1)
        s.cylinder((0.0, -4.0, 0.0), 3.0, 8.0, m)
        s.disk((0.0, 9.0, 0.0), 8.0, 0.1, m)
    return s


SCENES = {"mesh": lambda: scenes.sphere_mesh_scene(20000, seed=4), "lit": _lit, "shapes": scenes.shapes_scene,
          "instanced": lambda: _instanced(False), "instanced_shapes": lambda: _instanced(True)}
# width, height, spp, depth: one path; fewer paths than a wave; ragged against waves, groups and tiles; full
# tiles with more paths than the launch has lanes; one segment per path; long paths
SIZES = [(1, 1, 1, 8), (7, 3, 1, 4), (37, 29, 9, 8), (160, 96, 36, 6), (64, 64, 4, 1), (24, 16, 4, 60)]


@pytest.mark.parametrize("kind", sorted(SCENES))
def test_whole_paths_equal_stages(kind):
    s = SCENES[kind]()
    with Renderer(max_paths=1 << 20) as whole, Renderer(max_paths=1 << 20, extend_kernel=1) as staged:
        a, b = whole.upload(s), staged.upload(s)
        for rng in ("pcg", "minstd"):
            for w, h, spp, depth in SIZES:
                print("%s %s %dx%d %d spp depth %d" % (kind, rng, w, h, spp, depth), flush=True)
                rgb0, acc0, st0 = staged.render(b, w, h, spp, depth, seed=7, rng=rng)
                rgb1, acc1, st1 = whole.render(a, w, h, spp, depth, seed=7, rng=rng)
                assert np.array_equal(acc0, acc1, equal_nan=True)
                assert np.array_equal(rgb0, rgb1)
                for key in ("rays", "paths", "retraces", "light_pdf_tests"):
                    assert st0[key] == st1[key], key
                assert staged.counters()["exact_queries"] == whole.counters()["exact_queries"]
        if kind == "lit":
            assert st1["retraces"] > 0


def test_whole_paths_in_many_passes_and_sample_ranges():
    """A pass of 1,000 path ids cuts the request into pixel ranges of one sample, which no 8x8 tile order
    applies to (and the minstd stream into pixel ranges with all samples); a sample range alone."""
    s = scenes.sphere_mesh_scene(5000, seed=1)
    with Renderer(max_paths=1000, pass_paths=1000) as whole, Renderer(max_paths=1 << 18, extend_kernel=1) as staged:
        a, b = whole.upload(s), staged.upload(s)
        for rng, first, count in (("pcg", 0, 0), ("pcg", 3, 5), ("minstd", 0, 0)):
            _, acc0, st0 = staged.render(b, 48, 40, 9, 6, seed=5, rng=rng, sample_begin=first, sample_count=count)
            _, acc1, st1 = whole.render(a, 48, 40, 9, 6, seed=5, rng=rng, sample_begin=first, sample_count=count)
            assert np.array_equal(acc0, acc1, equal_nan=True)
            assert st0["rays"] == st1["rays"] and st0["paths"] == st1["paths"]
            assert whole.counters()["passes"] > 1


def test_whole_paths_in_a_batch():
    """Launches of different scenes and streams side by side on the renderer's streams."""
    kinds = sorted(SCENES)
    out = []
    for kw in (dict(), dict(sub_passes=4), dict(extend_kernel=1)):
        with Renderer(max_paths=1 << 20, **kw) as r:
            ids = [r.upload(SCENES[k]()) for k in kinds]
            jobs = [dict(sid=ids[i % len(ids)], width=40 + 9 * i, height=33 + 4 * i, spp=1 + 3 * i, max_depth=5, seed=i,
                         rng="minstd" if i % 3 == 2 else "pcg") for i in range(11)]
            res, st = r.render_batch(jobs)
            out.append(([acc for _, acc in res], st["rays"], st["paths"]))
    for accs, rays, paths in out[:2]:
        assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(accs, out[2][0]))
        assert (rays, paths) == out[2][1:]
