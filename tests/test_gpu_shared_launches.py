"""Short requests that share a whole-path launch (a batch's, and those waiting in the serving loop) and
large ones whose segments go over both lanes: images, sums and ray counts equal each request rendered
alone."""
import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, scenes

pytestmark = pytest.mark.gpu

# width, height, spp: one path; less, exactly and just over a wave's group; ragged; more than one launch
# takes (2^18 ids, so the next request starts another)
SHAPES = [(1, 1, 1), (7, 9, 1), (8, 8, 1), (13, 5, 1), (64, 64, 4), (37, 29, 9), (256, 256, 4), (300, 200, 9), (16, 16, 4),
          (129, 65, 16), (1, 64, 1), (64, 64, 16)]


def _check(r, jobs, got):
    for k, (j, (rgb, acc, rays)) in enumerate(zip(jobs, got)):
        rgb0, acc0, st0 = r.render(**j)
        assert np.array_equal(acc, acc0, equal_nan=True), k
        assert np.array_equal(rgb, rgb0), k
        assert rays is None or rays == st0["rays"], k


@pytest.mark.parametrize("rng", ["pcg", "minstd", "both"])
def test_short_requests_of_several_scenes(rng):
    with Renderer(max_paths=1 << 20) as r:
        sids = [r.upload(s) for s in (scenes.box_scene(), scenes.sphere_mesh_scene(5000, seed=1), scenes.shapes_scene(),
                                      scenes.instanced_scene(seed=2, n_instances=40, n_textures=2, tex_size=32, nu=12, nv=8, extent=10.0))]
        modes = ["pcg", "minstd"] if rng == "both" else [rng]
        jobs = [dict(sid=sids[(k // 3) % len(sids)], width=w, height=h, spp=n, max_depth=8, seed=k, rng=modes[k % len(modes)])
                for k, (w, h, n) in enumerate(SHAPES * 4)]
        imgs, _ = r.render_batch(jobs)
        _check(r, jobs, [(rgb, acc, None) for rgb, acc in imgs])
        ids = [r.submit(**j) for j in jobs]
        got = [r.wait(i, j["width"], j["height"]) for i, j in zip(ids, jobs)]
        _check(r, jobs, [(rgb, acc, st["rays"]) for rgb, acc, st in got])


@pytest.mark.parametrize("paths", [1 << 20, 3000])
def test_long_requests_over_both_lanes_among_short_ones(paths):
    """Requests of several segments (8 M paths; 1,500 ids a lane in the small pool), cancelled ones between."""
    big = (1200, 900, 9) if paths > 3000 else (90, 40, 4)
    with Renderer(max_paths=paths, pass_paths=0 if paths > 3000 else paths) as r:
        sid = r.upload(scenes.sphere_mesh_scene(20000, seed=4))
        jobs = [dict(sid=sid, width=w, height=h, spp=n, max_depth=6, seed=k, rng=m)
                for k, (w, h, n, m) in enumerate([(*big, "pcg"), (8, 8, 4, "pcg"), (*big, "minstd"), (*big, "pcg"), (64, 33, 4, "minstd")])]
        ids = [r.submit(**j) for j in jobs]
        dropped = r.submit(**dict(jobs[0], seed=99))
        r.cancel(dropped)
        got = [r.wait(i, j["width"], j["height"]) for i, j in zip(ids, jobs)]
        _check(r, jobs, [(rgb, acc, st["rays"]) for rgb, acc, st in got])


@pytest.mark.parametrize("config", [dict(extend_kernel=1, graphs=1), dict(extend_kernel=1, graphs=2), dict(bvh_width=2)])
def test_contexts_that_run_in_stages_serve_in_stages(config):
    """The open passes of the stages (enough iterations that captured ones are replayed) give what
    whole-path launches give."""
    s = scenes.sphere_mesh_scene(5000, seed=1)
    with Renderer(max_paths=1 << 16, pass_paths=1 << 18) as whole, Renderer(max_paths=1 << 16, pass_paths=1 << 18, **config) as r:
        a, b = whole.upload(s), r.upload(s)
        jobs = [dict(width=97, height=61, spp=9, max_depth=6, seed=k, rng=m) for k, m in enumerate(["pcg", "minstd", "pcg", "pcg"])]
        for _ in range(3):
            ids = [r.submit(b, **j) for j in jobs]
            got = [r.wait(i, j["width"], j["height"]) for i, j in zip(ids, jobs)]
            _check(whole, [dict(j, sid=a) for j in jobs], [(rgb, acc, st["rays"]) for rgb, acc, st in got])
