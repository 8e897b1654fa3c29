"""Raster windows from pixel boxes at their edges, against the oracle.

Triangles from a fraction of a pixel to a few windows across, placed over tile,
block and quad borders and over the target's right and lower edge, at every
sample count, with one wave and four per tile, in the deterministic and the
tagging mode, with and without clearing: IDs, depth bits, classes and fragment
counts must be equal.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _triangles(rng, n, W, H, size):
    """n triangles about `size` pixels across, half of them thin, centred on pixel positions near
    multiples of 16, 4 and 2 and near the far corner."""
    g = rng.choice([2, 4, 16], (n, 1))
    c = np.rint(rng.uniform(0, 1, (n, 2)) * np.array([W, H]) / g) * g + rng.uniform(-1.5, 1.5, (n, 2))
    c[::5] = np.array([W, H]) + rng.uniform(-3, 3, (len(c[::5]), 2))
    d = rng.uniform(-0.5, 0.5, (n, 3, 2)) * size
    d[1::2, :, 1] *= 0.05
    a = rng.uniform(0, 2 * np.pi, (n, 1))
    d = np.stack([d[..., 0] * np.cos(a) - d[..., 1] * np.sin(a), d[..., 0] * np.sin(a) + d[..., 1] * np.cos(a)], -1)
    ndc = (c[:, None] + d) * 2 / np.array([W, H]) - 1
    clip = np.concatenate([ndc, rng.uniform(0, 1, (n, 3, 1)), np.ones((n, 3, 1))], -1).reshape(-1, 4)
    return clip.astype(np.float32), np.arange(3 * n, dtype=np.int32)


@pytest.mark.parametrize("samples,threads,tagging", [(1, 256, False), (1, 64, False), (1, 256, True), (4, 256, False),
                                                     (8, 256, False)])
@pytest.mark.parametrize("size", [0.4, 1.5, 3.0, 5.0, 9.0, 24.0])
def test_windows_match_oracle(renderer_factory, samples, threads, tagging, size):
    r = renderer_factory()
    r.set_tuning(rasterTileThreads=threads)
    r.set_deterministic(not tagging)
    rng = np.random.default_rng(int(size * 10) + samples)
    for it, (W, H) in enumerate([(64, 48), (37, 51), (131, 66)]):
        clip, idx = _triangles(rng, [300, 700, 40][it], W, H, size)
        more, _ = _triangles(rng, 60, W, H, size)
        f = O.Frame().render(W, H, samples, clip, idx, tagging=tagging)
        g = O.Frame().render(W, H, samples, more, idx[:180], clear=False, depth_in=f.depth, tagging=tagging)
        r.set_target(W, H, samples)
        r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32)))
        r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
        print(f"[windows s={samples} t={threads} tagging={tagging} size={size} {W}x{H}]", flush=True)
        st = r.draw()
        ids, depth = r.visibility()
        assert np.array_equal(ids, f.ids)
        assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
        assert st["fragments"] == f.stats["fragments"] and st["coveredSamples"] == f.stats["covered_samples"]
        if samples == 1:
            assert np.array_equal(r.coverage_class(), f.cls)
        r.bind_geometry(more, idx[:180], np.eye(4, dtype=np.float32), clip_passthrough=True)
        st = r.draw(clear=False)
        _, depth = r.visibility()
        assert np.array_equal(depth.view(np.uint32), g.depth.view(np.uint32))
        assert st["coveredSamples"] == g.stats["covered_samples"]
