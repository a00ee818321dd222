"""The autotuner on whole-path launches: it may change the streams of a context only for what its trials can
show. On the CPU (hip_standin), where a launch takes as long as its paths are many and every measurement
is off by up to a hundredth."""
import pytest

from cortexraytracercuda_amd import Renderer, scenes
from hip_standin import standin, standin_lib  # noqa: F401


@pytest.mark.parametrize("rng", ["pcg", "minstd"])
@pytest.mark.parametrize("given,overlap,expected", [(0, 1, 2), (3, 1, 3), (0, 2, 2), (0, 4, 4), (1, 3, 3)])
def test_streams_change_only_for_a_gain(standin, rng, given, overlap, expected):
    standin.standin_overlap(overlap)
    with Renderer(max_paths=1 << 20, pass_paths=1 << 23, sub_passes=given) as r:
        sid = r.upload(scenes.box_scene())
        res = r.autotune(sid, 300, 200, 64, 4, rng=rng)
        assert res["sub_passes"] == expected
        # the stages' shape is as it was
        assert (res["max_paths"], res["grid_per_cu"], res["shade_grid_per_cu"], res["stack_lds"]) == (1 << 20, 24, 16, 16)
