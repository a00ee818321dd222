"""The serving loop's scheduler while launches run that do not end. On the CPU (hip_standin), where path
launches wait at a gate."""
import time

import numpy as np
import pytest

from cortexraytracercuda_amd import Renderer, _abi as A, scenes
from hip_standin import gate_closed, launches_that_ran, standin, standin_lib  # noqa: F401


def _until(what, seconds=10.0):
    end = time.monotonic() + seconds
    while time.monotonic() < end:
        if what():
            return True
        time.sleep(0.002)
    return False


def test_a_request_that_arrives_during_a_launch_takes_the_idle_lane(standin):
    with Renderer(max_paths=1 << 15, pass_paths=1 << 16) as r:
        sid = r.upload(scenes.box_scene())
        with gate_closed(standin):
            first = r.submit(sid, 64, 64, 4, 3, seed=1)
            assert _until(lambda: standin.standin_launches() == 1)
            time.sleep(0.05)   # the scheduler has nothing left to do
            second = r.submit(sid, 8, 8, 4, 3, seed=2)
            assert _until(lambda: standin.standin_launches() == 2)
            assert not r.poll(first) and not r.poll(second)
        for i, w in ((first, 64), (second, 8)):
            assert r.wait(i, w, w)[2]["rays"] == w * w * 4


def test_a_waiting_request_is_cancelled_during_a_launch(standin):
    with Renderer(max_paths=1 << 15, pass_paths=1 << 16) as r:
        r.wait(r.submit(r.upload(scenes.box_scene()), 8, 8, 1, 2), 8, 8)
        held = sum(r.memory()[k] for k in ("reserved", "scenes"))
    with Renderer(max_paths=1 << 15, pass_paths=1 << 16, hbm_budget=held + 64 * 64 * 19 + 4096) as r:
        sid = r.upload(scenes.box_scene())
        with gate_closed(standin):
            first = r.submit(sid, 64, 64, 4, 3, seed=1)
            assert _until(lambda: standin.standin_launches() == 1)
            time.sleep(0.05)
            second = r.submit(sid, 64, 60, 4, 3, seed=2)   # does not fit beside the first
            r.cancel(second)
            assert _until(lambda: r.poll(second))
            with pytest.raises(A.CrtError, match="cancelled"):
                r.wait(second, 64, 60)
            assert not r.poll(first)
        assert r.wait(first, 64, 64)[2]["rays"] == 64 * 64 * 4


@pytest.mark.parametrize("w,h,spp,cap", [(16, 12, 1, 0), (16, 12, 64, 0), (16, 12, 81, 0), (31, 17, 1024, 0), (8, 4, 65536, 0),
                                         (31, 17, 400, 200), (64, 33, 144, 1000)])
def test_reference_streams_are_served_in_bounded_launches(standin, w, h, spp, cap):
    """A pixel's samples go on from one launch to the next, on whichever lane: sums equal the blocking
    render's. With `cap` path ids a lane, pixels are cut as well."""
    with Renderer(max_paths=max(cap * 2, 1 << 12), pass_paths=max(cap * 2, 1 << 24)) as r:
        sid = r.upload(scenes.box_scene())
        rgb, acc, st = r.render(sid, w, h, spp, 3, seed=5, rng="minstd")
        alone = len(launches_that_ran(standin))
        others = [r.submit(sid, 20, 10, 9, 3, seed=k, rng=m) for k, m in enumerate(("pcg", "minstd"))]
        mine = r.submit(sid, w, h, spp, 3, seed=5, rng="minstd")
        srgb, sacc, sst = r.wait(mine, w, h)
        for k in others:
            r.wait(k, 20, 10)
        assert np.array_equal(sacc, acc) and np.array_equal(srgb, rgb) and sst["rays"] == st["rays"]
        for l in launches_that_ran(standin)[alone:]:
            if l["mode"] == A.CRT_RNG_MINSTD:
                assert l["samples"] <= 64 and l["paths"] <= 1 << 24


def test_reference_streams_over_many_pixels_are_served_in_bounded_launches(standin):
    with Renderer(max_paths=1 << 12, pass_paths=1 << 24) as r:
        sid = r.upload(scenes.box_scene())
        _, acc, _ = r.render(sid, 700, 500, 81, 3, seed=5, rng="minstd")
        alone = len(launches_that_ran(standin))
        _, sacc, _ = r.wait(r.submit(sid, 700, 500, 81, 3, seed=5, rng="minstd"), 700, 500)
        assert np.array_equal(sacc, acc)
        ran = launches_that_ran(standin)[alone:]
        assert len(ran) == 4 and max(l["paths"] for l in ran) <= 1 << 24


def test_a_long_reference_stream_is_not_enqueued_far_ahead(standin):
    """Sample ranges take their time however small the image is: each lane has one of them, and a request
    that arrives takes its turn behind those."""
    with Renderer(max_paths=1 << 12, pass_paths=1 << 22, serve_small_paths=1000) as r:
        sid = r.upload(scenes.box_scene())
        with gate_closed(standin):
            first = r.submit(sid, 32, 20, 4096, 3, seed=1, rng="minstd")
            assert _until(lambda: standin.standin_launches() == 2)
            second = r.submit(sid, 8, 8, 4, 3, seed=2)
            time.sleep(0.1)
            assert standin.standin_launches() == 2
        r.wait(second, 8, 8)
        assert launches_that_ran(standin)[2]["mode"] == A.CRT_RNG_PCG
        r.wait(first, 32, 20)
