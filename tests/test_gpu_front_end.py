"""Geometry kernel and binning at the edges of their cases, against the oracle.

One renderer draws one scene after another, so that every draw starts from the
counters the previous one left: triangle counts around the wave and workgroup
sizes, rectangles of one, two to four, up to eight, up to the deferral
threshold and more tiles, triangles across w = 0 with small and screen-sized
fans, and render targets of changing tile counts.  Integer results and depth
bits must be equal.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TARGETS = [(33, 17), (256, 256), (257, 129), (640, 400)]


def _triangles(rng, n, W, H, extent):
    """n front- or back-facing triangles about `extent` tiles across; every eighth crosses w = 0."""
    c = rng.uniform(-1, 1, (n, 1, 2))
    d = rng.uniform(-1, 1, (n, 3, 2)) * (16.0 * extent / np.array([W, H]))
    w = rng.uniform(0.5, 2.0, (n, 3, 1))
    w[::8, 0] = -rng.uniform(0.2, 1.0, (len(w[::8]), 1))
    z = rng.uniform(0, 1, (n, 3, 1))
    clip = np.concatenate([(c + d) * np.abs(w), z * np.abs(w), w], -1).reshape(-1, 4)
    return clip.astype(np.float32), np.arange(3 * n, dtype=np.int32)


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("extent", [0.2, 1.0, 2.5, 8.0, 40.0])
def test_counts_and_rectangles(renderer_factory, samples, extent):
    r = renderer_factory()
    rng = np.random.default_rng(int(extent * 10) + samples)
    for it, n in enumerate([1, 63, 64, 65, 255, 256, 257, 1025, 2]):
        W, H = TARGETS[it % len(TARGETS)]
        clip, idx = _triangles(rng, n, W, H, extent)
        f = O.Frame().render(W, H, samples, clip, idx)
        r.set_target(W, H, samples)
        r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
        r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32)))
        print(f"[front end s={samples} extent={extent} n={n} {W}x{H}]", flush=True)
        for _ in range(2):
            st = r.draw()
            ids, depth = r.visibility()
            assert np.array_equal(ids, f.ids)
            assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
            assert st["fragments"] == f.stats["fragments"]
            assert st["coveredSamples"] == f.stats["covered_samples"]
            assert st["assembledTriangles"] == f.stats["assembled_triangles"]


def test_bin_list_overflow_leaves_clean_counters(renderer_factory):
    """A bin list too small for the draw is grown and drawn again; the next, smaller draw is unaffected."""
    r = renderer_factory()
    rng = np.random.default_rng(3)
    W, H = 640, 400
    big, bi = _triangles(rng, 3000, W, H, 20.0)
    small, si = _triangles(rng, 50, W, H, 1.0)
    r.set_target(W, H, 1)
    r.set_tuning(binCapacity=4096)
    for clip, idx in ((big, bi), (small, si)):
        f = O.Frame().render(W, H, 1, clip, idx)
        r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
        r.bind_fragment_program(scenes.Scene("t", W, H, 1, clip, idx, np.eye(4, dtype=np.float32)))
        st = r.draw()
        ids, depth = r.visibility()
        print(f"[bin overflow] retries {st['retries']} entries {st['binEntries']}", flush=True)
        assert np.array_equal(ids, f.ids)
        assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
