"""Depth functions drawn through order-independent keys, against the oracle's fold in primitive order.

LESS_OR_EQUAL, GREATER, GREATER_OR_EQUAL and ALWAYS on cleared targets, where
ties and special values decide: depths from a few values with both zeros and
the clear depth itself among them, the first primitive drawn at the clear
depth, lists long enough to be cut into parts, and tiles with NaN depths, whose
result depends on the order after all.  IDs, classes and depth bits must be
equal (a NaN only has to be one: its payload is the machine's).
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _scene(rng, n, W, H, zs, nan):
    c = rng.uniform(-1, 1, (n, 1, 2))
    xy = c + rng.uniform(-0.4, 0.4, (n, 3, 2))
    xy[0] = [[-1, -1], [1, -1], [0, 1]]
    z = np.repeat(rng.choice(zs, (n, 1, 1)), 3, 1)
    if nan:
        z[rng.integers(0, n, 3)] = np.nan
    clip = np.concatenate([xy, z, np.ones((n, 3, 1))], -1).reshape(-1, 4).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    flip = rng.random(n) < 0.5
    flip[0] = False
    idx[flip] = idx[flip][:, ::-1]
    both = np.concatenate([idx, idx[:, ::-1]])  # either winding survives the cull
    return clip, np.ascontiguousarray(both.reshape(-1))


@pytest.mark.parametrize("samples,threads,tagging", [(1, 256, False), (1, 64, False), (1, 256, True), (4, 256, False),
                                                     (8, 256, False)])
@pytest.mark.parametrize("func", [3, 4, 6, 7])
def test_keys_match_the_fold(renderer_factory, func, samples, threads, tagging):
    r = renderer_factory()
    r.set_tuning(rasterTileThreads=threads, rasterPartEntries=256)
    r.set_deterministic(not tagging)
    r.set_depth_func(func)
    rng = np.random.default_rng(10 * func + samples)
    for it, (n, nan) in enumerate([(60, False), (900, False), (200, True)]):
        W, H = [(70, 45), (32, 32), (64, 33)][it]
        for clear in (0.5, 0.0, 1.0):
            clip, idx = _scene(rng, n, W, H, [0.0, -0.0, 0.25, 0.5, 1.0], nan)
            clip[:3, 2] = clear
            f = O.Frame().render(W, H, samples, clip, idx, depth_func=func, clear_depth=clear, tagging=tagging)
            r.set_target(W, H, samples)
            r.set_clear_values(depth=clear)
            r.bind_geometry(clip, idx, np.eye(4, dtype=np.float32), clip_passthrough=True)
            r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, np.eye(4, dtype=np.float32)))
            print(f"[keys func={func} s={samples} t={threads} tagging={tagging} n={n} nan={nan} clear={clear}]", flush=True)
            for _ in range(2):
                st = r.draw()
                ids, depth = r.visibility()
                assert np.array_equal(ids, f.ids)
                same = (depth.view(np.uint32) == f.depth.view(np.uint32)) | (np.isnan(depth) & np.isnan(f.depth))
                assert same.all()
                assert st["fragments"] == f.stats["fragments"] and st["coveredSamples"] == f.stats["covered_samples"]
                if samples == 1:
                    assert np.array_equal(r.coverage_class(), f.cls)
