"""The ordered traversal at the edges of its lists, against the oracle's fold in primitive order.

List lengths around a sorting wave (64), a chunk of records (128), one, four and
eight keys per thread (256, 1024, 2048) and several sorted windows (above 2048);
triangles of a pixel, of one window, of several blocks of the grid, of more than
four windows, and such that cover whole tiles; targets that end inside a tile.
IDs, classes, depth bits and blended FP32 colours must be equal.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

from test_oracle_pins import BLENDS

pytestmark = pytest.mark.gpu

COUNTS = (1, 63, 64, 65, 127, 129, 255, 257, 1000, 1025, 2047, 2049, 4500)


def _scene(rng, n, W, H):
    size = rng.choice([1.0, 3.0, 6.0, 12.0, 60.0], n, p=[0.5, 0.2, 0.15, 0.1, 0.05])[:, None, None]
    c = rng.uniform(0, 1, (n, 1, 2)) * [W, H]
    px = c + rng.uniform(-1, 1, (n, 3, 2)) * size
    z = rng.choice([0.25, 0.5, 0.5, 0.75], (n, 1, 1)) + rng.uniform(0, 0.01, (n, 3, 1))
    clip = np.concatenate([px / [W, H] * 2 - 1, z, np.ones((n, 3, 1))], -1).reshape(-1, 4).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    e1, e2 = px[:, 1] - px[:, 0], px[:, 2] - px[:, 0]
    idx[e1[:, 0] * e2[:, 1] < e1[:, 1] * e2[:, 0]] = idx[e1[:, 0] * e2[:, 1] < e1[:, 1] * e2[:, 0]][:, ::-1]
    idx[:, :] = idx if rng.random() < 0.5 else idx[:, ::-1]
    return clip, np.ascontiguousarray(np.concatenate([idx, idx[::2, ::-1]]).reshape(-1))  # some of either winding


def _bind(r, W, H, samples, clip, idx):
    r.set_target(W, H, samples)
    s = scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32), program=scenes.PROGRAM_FLAT_ALPHA)
    r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
    r.bind_fragment_program(s)


@pytest.mark.parametrize("samples,func,tagging", [(1, 5, False), (1, 4, False), (1, 5, True), (4, 5, False),
                                                  (8, 5, False)])
def test_fold_matches_oracle(renderer_factory, samples, func, tagging):
    r = renderer_factory()
    r.set_deterministic(not tagging)
    r.set_depth_func(func)
    for n in COUNTS:
        rng = np.random.default_rng(n)
        W, H = [(16, 16), (21, 13)][n % 2]
        clip, idx = _scene(rng, n, W, H)
        _bind(r, W, H, samples, clip, idx)
        print(f"[ordered lists s={samples} func={func} tagging={tagging} n={n}]", flush=True)
        st = r.draw()
        ids, depth = r.visibility()
        f = O.Frame().render(W, H, samples, clip, idx, depth_func=func, tagging=tagging)
        assert np.array_equal(ids, f.ids)
        assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
        assert st["fragments"] == f.stats["fragments"] and st["coveredSamples"] == f.stats["covered_samples"]
        if samples == 1:
            assert np.array_equal(r.coverage_class(), f.cls)


def test_blend_matches_oracle(renderer_factory):
    r = renderer_factory()
    r.set_depth_func(7)
    r.set_blend(BLENDS[0])
    for n in COUNTS:
        W, H = [(16, 16), (21, 13)][n % 2]
        clip, idx = _scene(np.random.default_rng(n), n, W, H)
        _bind(r, W, H, 1, clip, idx)
        print(f"[ordered lists blend n={n}]", flush=True)
        r.draw()
        got = r.color_f32()
        f = O.Frame().render_blend(W, H, clip, idx, BLENDS[0], depth_func=7)
        assert np.array_equal(r.visibility()[0], f.ids)
        assert np.array_equal(got.view(np.uint32), f.rgba.view(np.uint32))
