"""Clipping and tile plan of a single view in one launch, against the oracle.

Triangles that cross w = 0, triangles over hundreds of tiles, both and neither, on targets of fewer tile
plan workgroups than clipping shares, about as many, and more (17424 tiles: 69 of 256 tiles); the third draw
repeats the first, after one that left other counts.  IDs, depth bits and statistics must be equal.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _scene(rng, clipped, big):
    n = 600
    c = rng.uniform(-0.9, 0.9, (n, 1, 3)).astype(np.float32)
    half = np.full((n, 1, 1), 0.04, np.float32)
    half[:big] = 1.5
    v = np.ones((n, 3, 4), np.float32)
    v[..., :3] = c + half * rng.uniform(-1, 1, (n, 3, 3)).astype(np.float32)
    v[..., 2] = 0.5 + 0.4 * rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    w = rng.uniform(0.5, 2.0, (n, 3)).astype(np.float32)
    v[..., :3] *= w[..., None]
    v[..., 3] = w
    v[n - clipped:, 0, 3] = -0.3  # one vertex behind the eye
    idx = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    idx = np.concatenate([idx, idx[:, ::-1]])
    return v.reshape(-1, 4), np.ascontiguousarray(idx.reshape(-1))


@pytest.mark.parametrize("W,H", [(33, 17), (640, 480), (2100, 2100)])
@pytest.mark.parametrize("clipped,big", [(0, 0), (200, 0), (0, 6), (200, 6)])
def test_clip_plan(renderer_factory, W, H, clipped, big):
    clip, idx = _scene(np.random.default_rng(41 + clipped + big), clipped, big)
    clip2, idx2 = _scene(np.random.default_rng(5), 100, 3)
    r = renderer_factory()
    r.set_target(W, H, 1)
    f = O.Frame().render(W, H, 1, clip, idx)
    for k, (c, i) in enumerate([(clip, idx), (clip2, idx2), (clip, idx)]):
        r.bind_geometry(c, i, np.eye(4, dtype=np.float32), clip_passthrough=True)
        r.bind_fragment_program(scenes.Scene("t", W, H, 1, c, i, np.eye(4, dtype=np.float32)))
        print(f"[clip plan {W}x{H} clipped={clipped} big={big} draw {k}]", flush=True)
        st = r.draw()
        if k == 1:
            continue
        ids, depth = r.visibility()
        assert np.array_equal(ids, f.ids)
        assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
        assert st["fragments"] == f.stats["fragments"] and st["coveredSamples"] == f.stats["covered_samples"]
        assert (st["clippedTriangles"] > 0) == (clipped > 0)
