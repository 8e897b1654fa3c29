"""A no-allocation draw between an asynchronous draw and the call that waits for it.

The waiting call must tell the asynchronous draw's statistics and overflow, whether its
counters were reduced with the draw (LESS) or are reduced when asked for (NOT_EQUAL), and
nothing of the no-allocation draw's.
"""
import ctypes as C

import numpy as np
import pytest

import ifrit_hip
from ifrit_hip import IfritError, scenes

from test_gpu_kept_slots import EYE, _bind, _overlay
from test_gpu_shade_order import _scene
from test_zz_no_alloc import _DeviceArrays

pytestmark = pytest.mark.gpu

W, H = 320, 201
COUNTS = ("inputTriangles", "assembledTriangles", "clippedTriangles", "binEntries", "fragments", "coveredSamples")


def _noalloc(r, clip, idx, samples, error=None):
    dev = _DeviceArrays()
    try:
        depth = dev.put(np.zeros(r.width * r.height * samples, np.float32))
        d = ifrit_hip.NoAllocDraw(dev.put(clip), clip.shape[1], clip.shape[0], dev.put(idx), idx.size, None, depth, None)
        r.L.iftrDrawNoAlloc(r.h, C.byref(d))
        if error is None:
            r._check()
        else:
            with pytest.raises(IfritError, match=error):
                r._check()
    finally:
        dev.free()


@pytest.mark.parametrize("func", [1, 5])
def test_statistics_are_the_asynchronous_draws(renderer_factory, func):
    r = renderer_factory()
    clip, idx = _scene(np.random.default_rng(func), W, H, 2000)
    over, oi = _overlay()
    r.set_depth_func(func)
    r.set_target(W, H, 1)
    _bind(r, W, H, 1, clip, idx)
    want = r.draw()
    assert want["fragments"] > 1000
    print(f"[no-allocation draw between, func={func}]", flush=True)
    r.draw_async()
    _noalloc(r, over, oi, 1)
    assert r.stats()["inputTriangles"] == oi.size // 3
    r.synchronize()
    got = r.stats()
    assert [got[k] for k in COUNTS] == [want[k] for k in COUNTS]


def test_overflow_is_reported(renderer_factory):
    r = renderer_factory()
    clip, idx = _scene(np.random.default_rng(3), W, H, 5600)
    over, oi = _overlay()
    r.set_target(W, H, 1)
    _bind(r, W, H, 1, clip, idx)
    want = r.draw()
    r.set_tuning(binCapacity=4096)
    print("[no-allocation draw between, overflow]", flush=True)
    r.draw_async()
    _noalloc(r, over, oi, 1)
    with pytest.raises(IfritError, match="binning buffers"):
        r.synchronize()
    assert r.tuning()["binCapacity"] > want["binEntries"]


def test_overflow_of_the_no_allocation_draw_stays_its_own(renderer_factory):
    r = renderer_factory()
    clip, idx = _scene(np.random.default_rng(3), 1024, 1024, 500)
    r.set_target(1024, 1024, 1)
    _bind(r, 1024, 1024, 1, clip, idx)
    want, cap = r.draw(), r.tuning()["binCapacity"]
    big = np.array([[-1, -1, 0.5, 1], [3, -1, 0.5, 1], [-1, 3, 0.5, 1]], np.float32)
    bi = np.tile(np.array([0, 1, 2, 2, 1, 0], np.int32), 300)  # 300 face the eye, 4096 tiles each
    print("[no-allocation draw between, its own overflow]", flush=True)
    r.draw_async()
    _noalloc(r, big, bi, 1, "overflowed its scratch buffers")
    r.synchronize()
    got = r.stats()
    assert [got[k] for k in COUNTS] == [want[k] for k in COUNTS]
    assert r.tuning()["binCapacity"] == cap
