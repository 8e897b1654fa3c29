"""Shading in the tile plan's order: every pixel of every tile exactly once, whatever its list.

Flat-coloured triangles whose lists are empty, short, long and longer than a part, in
one target that ends inside a tile; waves per 8x8 sub-tile, per tile and per four
tiles; a clear colour, a scissor, and a second draw without clear.  The colour is the
mean over the samples of a hash of the primitive ID that the visibility holds, or the
clear colour; a sum of up to eight products of values in [0, 1] and its division
differ by at most 16 roundings, 16 * 2^-24 < 1e-6.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _scene(rng, W, H, dense):
    """Triangles of a few pixels: none in the left columns, `dense` of them per tile on the right."""
    c = np.concatenate([rng.uniform([W / 4, 0], [W, H], (400, 2)), rng.uniform([W * 3 / 4, 0], [W, H], (dense, 2))])
    n = len(c)
    ang = rng.uniform(0, 2 * np.pi, (n, 1)) + np.array([0, 2.1, 4.2])
    px = c[:, None] + rng.uniform(1.0, 4.0, (n, 1, 1)) * np.stack([np.cos(ang), np.sin(ang)], -1)
    z = np.repeat(rng.uniform(0.1, 0.9, (n, 1, 1)), 3, 1)
    clip = np.concatenate([px / [W, H] * 2 - 1, z, np.ones((n, 3, 1))], -1).reshape(-1, 4).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    return clip, np.ascontiguousarray(np.concatenate([idx, idx[:, ::-1]]).reshape(-1))


def _flat(ids, clear):
    prims, at = np.unique(ids, return_inverse=True)
    h = np.array([O.flat_hash(int(p)) for p in prims], np.uint32)[at].reshape(ids.shape)
    c = np.stack([h & 255, (h >> np.uint32(8)) & 255, (h >> np.uint32(16)) & 255, np.full_like(h, 255)], -1) / 255.0
    c[ids == 0xFFFFFFFF] = clear
    return c


@pytest.mark.parametrize("samples", [1, 4, 8])
@pytest.mark.parametrize("tile", [8, 16, 32])
def test_every_pixel_shaded_once(renderer_factory, tile, samples):
    r = renderer_factory()
    r.set_tuning(shadeTile=tile)
    r.set_float_output(True)
    clear = np.array([0.25, 0.5, 0.75, 1.0])
    r.set_clear_values(clear, 1.0)
    rng = np.random.default_rng(tile + samples)
    for W, H, dense, scissor in [(150, 77, 9000, False), (16, 16, 0, False), (97, 40, 300, True)]:
        clip, idx = _scene(rng, W, H, dense)
        r.set_target(W, H, samples)
        r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
        r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32),
                                             program=scenes.PROGRAM_FLAT))
        r.set_scissors([], False)
        print(f"[shade order tile={tile} s={samples} {W}x{H} dense={dense} scissor={scissor}]", flush=True)
        r.draw()
        want = _flat(r.visibility()[0].reshape(H, W, samples), clear).mean(2)
        assert np.abs(r.color_f32().reshape(H, W, 4) - want).max() < 1e-6
        r.draw(clear=False)  # the same triangles: nothing passes, nothing changes
        assert np.abs(r.color_f32().reshape(H, W, 4) - want).max() < 1e-6
        if scissor:
            before = r.color_f32().reshape(H, W, 4)
            r.set_clear_values((1.0, 0.0, 0.5, 0.0), 1.0)
            r.set_scissors([(20.0, 9.0, 30.0, 20.0)])
            r.draw()
            y, x = np.mgrid[:H, :W]
            inside = (x >= 20) & (x <= 50) & (y >= 9) & (y <= 29)
            got = r.color_f32().reshape(H, W, 4)
            want2 = _flat(r.visibility()[0].reshape(H, W, samples), np.array([1.0, 0.0, 0.5, 0.0])).mean(2)
            assert np.array_equal(got[~inside], before[~inside])
            assert np.abs(got - want2)[inside].max() < 1e-6
            r.set_clear_values(clear, 1.0)
