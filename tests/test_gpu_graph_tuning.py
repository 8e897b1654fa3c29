"""A replayed graph follows the threads per tile: the raster's grid and the layout of its statistics do."""
import numpy as np
import pytest

from test_gpu_kept_slots import _bind
from test_gpu_shade_order import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("func", [1, 5])
def test_threads_per_tile_change_between_replays(renderer_factory, func):
    r = renderer_factory()
    W, H = 320, 201
    clip, idx = _scene(np.random.default_rng(func), W, H, 2000)
    r.set_depth_func(func)
    r.set_target(W, H, 1)
    _bind(r, W, H, 1, clip, idx)
    want, ids = r.draw(), r.visibility()[0]
    r.set_graph_mode(True)
    for threads in (64, 256, 64, 256):
        r.set_tuning(rasterTileThreads=threads)
        print(f"[graph func={func} threads={threads}]", flush=True)
        for _ in range(2):
            got = r.draw()
            assert got["fragments"] == want["fragments"] and got["coveredSamples"] == want["coveredSamples"]
            assert np.array_equal(r.visibility()[0], ids)
