"""The key raster's wide and narrow passes, against the oracle.

42000 triangles are wide passes for the default grid and narrow ones for a grid of one
workgroup per compute unit (320 * 128 = 40960 triangles on 256 of them).  Lists of
more than one pass and of more than one part; IDs, classes and depth bits must be
equal.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

from test_gpu_ordered_lists import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples", [1, 4, 8])
@pytest.mark.parametrize("func", [1, 3])
def test_wide_and_narrow_passes(renderer_factory, func, samples):
    W, H = 250, 141
    clip, idx = _scene(np.random.default_rng(7 + samples), 28000, W, H)  # half of them in either winding too
    assert idx.size // 3 == 42000
    f = O.Frame().render(W, H, samples, clip, idx, depth_func=func)
    r = renderer_factory()
    r.set_depth_func(func)
    r.set_target(W, H, samples)
    r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
    r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32)))
    for groups in (4, 1):
        r.set_tuning(rasterGroupsPerCU=groups)
        print(f"[raster passes s={samples} func={func} groups={groups}]", flush=True)
        st = r.draw()
        ids, depth = r.visibility()
        assert np.array_equal(ids, f.ids)
        assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
        assert st["fragments"] == f.stats["fragments"] and st["coveredSamples"] == f.stats["covered_samples"]
        if samples == 1:
            assert np.array_equal(r.coverage_class(), f.cls)
