"""Binning where a scatter wave takes several geometry waves (more than 8192 of them in the batch).

66 views of 61440 triangles (960 geometry waves each, 63360 in all, three at a time with
a remainder) and 9 views (8640, two at a time): IDs, depth bits and statistics of some
views must be those of the view drawn alone, where a wave takes one.
"""
import numpy as np
import pytest

from ifrit_hip import scenes

from test_gpu_batch import _alone, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [9, 66])
def test_batch_equals_views_alone(renderer_factory, count):
    s = scenes.config2(width=64, height=64, samples=1, spheres=12, level=4, tex_size=16, host_textures=True)
    assert s.indices.size == 3 * 61440
    base = scenes.config4_views(seed=3, cascade_size=100, cube_size=40, cameras=6, max_size=(90, 70), min_size=24)
    views = [base[i % len(base)] for i in range(count)]
    r = renderer_factory()
    r.load_scene(s)
    r.set_views(views)
    st = r.draw()
    got = {i: (*r.view_visibility(i), r.view_color(i) if views[i]["shade"] else None)
           for i in {0, 5, 8, count // 2, count - 1}}
    assert st["assembledTriangles"] > 0
    alone = renderer_factory()
    alone.load_scene(s)
    for i, out in sorted(got.items()):
        _same(out, _alone(alone, s, views[i]), f"scatter regions {count} views, view {i}")
