"""Primitive IDs that the no-allocation draw's raster writes itself, against the ordinary draw's.

Per sample count: the key raster (LESS), general keys with tiles drawn again for
their NaN depths (LESS_OR_EQUAL) and the ordered fold (NOT_EQUAL); lists cut into
parts and merged; targets whose rows are whole 16-byte words and such that are
not, ID arrays on and off a 16-byte line, a scissor, with and without colour.
IDs and depth bits must be equal (a NaN only has to be one), and so must what lies
outside the scissor and what surrounds the IDs.
"""
import ctypes as C

import numpy as np
import pytest

from ifrit_hip import scenes

from test_gpu_depth_keys import _scene
from test_zz_no_alloc import _DeviceArrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples", [1, 4, 8])
@pytest.mark.parametrize("func", [1, 3, 5])
def test_ids_match_draw(renderer_factory, func, samples):
    import ifrit_hip

    r = renderer_factory()
    r.set_tuning(rasterPartEntries=256)
    r.set_depth_func(func)
    rng = np.random.default_rng(100 * func + samples)
    for W, H, n, shift, scissor, shade in [(64, 48, 900, 0, False, False), (70, 45, 900, 1, False, True),
                                           (64, 33, 60, 1, False, False), (70, 45, 300, 0, True, True)]:
        clip, idx = _scene(rng, n, W, H, [0.25, 0.5, 0.75], func == 3)
        r.set_target(W, H, samples)
        r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
        r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32),
                                             program=scenes.PROGRAM_FLAT))
        r.set_scissors([(5.0, 3.0, 31.0, 20.0)] if scissor else [])
        print(f"[ids func={func} s={samples} {W}x{H} n={n} shift={shift} scissor={scissor} shade={shade}]", flush=True)
        r.draw()
        want, wantz = r.visibility()
        inside = np.ones((H, W), bool)
        if scissor:
            y, x = np.mgrid[:H, :W]
            inside = (x >= 5) & (x <= 36) & (y >= 3) & (y <= 23)
        inside = np.repeat(inside.reshape(-1), samples)
        dev = _DeviceArrays()
        try:
            buf = np.full(W * H * samples + 8, 0x5A5A5A5A, np.uint32)
            z0 = np.full(W * H * samples, -7.0, np.float32)
            c0 = np.zeros((H, W, 4), np.uint8)
            v, i = dev.put(clip), dev.put(idx)
            ids, depth, rgba = dev.put(buf), dev.put(z0), dev.put(c0) if shade else None
            d = ifrit_hip.NoAllocDraw(v, clip.shape[1], clip.shape[0], i, idx.size, C.c_void_p(ids.value + 4 * shift),
                                      depth, rgba)
            r.L.iftrDrawNoAlloc(r.h, C.byref(d))
            r._check()
            got, z = dev.get(ids, buf), dev.get(depth, z0)
        finally:
            dev.free()
        body = got[shift:shift + want.size]
        assert np.array_equal(body[inside], want.reshape(-1)[inside])
        wz = wantz.reshape(-1)
        assert ((z.view(np.uint32) == wz.view(np.uint32)) | (np.isnan(z) & np.isnan(wz)))[inside].all()
        assert (body[~inside] == 0x5A5A5A5A).all() and (z[~inside] == -7.0).all()
        assert (got[:shift] == 0x5A5A5A5A).all() and (got[shift + want.size:] == 0x5A5A5A5A).all()
