"""Forms of whole-path launches beside those of the other tests, each against the same requests rendered
alone or in stages: shared launches whose paths pass a visible spot light, refilled waves on a tree built
on the device, and reference streams that are served in several sample ranges."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


def _lit(s):
    s.omni_light((0.55, 0.45, -0.3), 0.12, rgb=(1.0, 0.8, 0.6), intensity=6.0, invisible=False)
    s.spot_light((0.0, 0.0, 0.8), (0.2, -1.0, 0.1), 35.0, 4.0, 0.3, rgb=(0.6, 0.8, 1.0), intensity=20.0, invisible=False)
    return s


@pytest.mark.parametrize("rng", ["pcg", "minstd"])
def test_shared_launches_that_pass_a_spot_light(rng):
    """Paths that carry the light's white on keep it in their radiance slots, which a shared launch counts
    from each request's own first id."""
    with Renderer(max_paths=1 << 20, extend_kernel=1) as staged, Renderer(max_paths=1 << 20) as r:
        make = (lambda: _lit(scenes.box_scene()), lambda: _lit(scenes.sphere_mesh_scene(3000, seed=2)))
        a, b = [staged.upload(m()) for m in make], [r.upload(m()) for m in make]
        jobs = [dict(width=w, height=h, spp=n, max_depth=6, seed=k, rng=rng)
                for k, (w, h, n) in enumerate([(31, 17, 4), (8, 8, 1), (64, 40, 9), (5, 3, 1), (33, 65, 4), (16, 16, 16)])]
        alone = [staged.render(a[k % 2], **j) for k, j in enumerate(jobs)]
        assert all(st["retraces"] > 0 for _, _, st in alone[2:3])
        jobs = [dict(j, sid=b[k % 2]) for k, j in enumerate(jobs)]
        res, st = r.render_batch(jobs)
        assert st["rays"] == sum(x[2]["rays"] for x in alone)
        ids = [r.submit(**j) for j in jobs]
        for k, (rgb, acc, _) in enumerate(alone):
            assert np.array_equal(res[k][1], acc, equal_nan=True) and np.array_equal(res[k][0], rgb), k
            srgb, sacc, sst = r.wait(ids[k], jobs[k]["width"], jobs[k]["height"])
            assert np.array_equal(sacc, acc, equal_nan=True) and np.array_equal(srgb, rgb) and sst["rays"] == alone[k][2]["rays"], k


@pytest.mark.parametrize("make", [lambda: _lit(scenes.sphere_mesh_scene(60000, seed=4)), lambda: scenes.large_scene(levels=6, n_spheres=200)])
def test_refilled_waves_on_a_device_built_tree(make):
    s = make()
    with Renderer(bvh_builder="device") as r, Renderer(bvh_builder="device", extend_kernel=1) as staged:
        a, b = r.upload(s), staged.upload(s)
        assert r.info(a)["builder"] == "device" and r.info(a)["num_nodes"] >= 1 << 14
        (rgb0, acc0, st0), (rgb1, acc1, st1) = [x.render(sid, 1021, 771, 9, 8, seed=3) for x, sid in ((r, a), (staged, b))]
        assert np.array_equal(acc0, acc1, equal_nan=True) and np.array_equal(rgb0, rgb1)
        assert all(st0[k] == st1[k] for k in ("rays", "paths", "retraces", "light_pdf_tests"))


@pytest.mark.parametrize("w,h,spp,paths", [(33, 21, 64, 0), (33, 21, 81, 0), (64, 48, 400, 0), (90, 40, 144, 3000)])
def test_reference_streams_over_several_sample_ranges(w, h, spp, paths):
    """More than 64 samples go over several launches and both lanes; with 1,500 ids a lane so do the pixels."""
    with Renderer(max_paths=paths or 1 << 20, pass_paths=paths) as r:
        sid = r.upload(_lit(scenes.sphere_mesh_scene(3000, seed=2)))
        other = [r.submit(sid, 40, 30, 4, 4, seed=k) for k in range(3)]
        mine = [r.submit(sid, w, h, spp, 5, seed=k, rng="minstd") for k in range(2)]
        for i in other:
            r.wait(i, 40, 30)
        for k, i in enumerate(mine):
            rgb, acc, st = r.wait(i, w, h)
            rgb0, acc0, st0 = r.render(sid, w, h, spp, 5, seed=k, rng="minstd")
            assert np.array_equal(acc, acc0, equal_nan=True) and np.array_equal(rgb, rgb0) and st["rays"] == st0["rays"]
