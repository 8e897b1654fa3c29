"""The ordered traversal's accepted blocks at the low corner of a pixel box, against the oracle.

A triangle clipped to a tile, or to one of its halves, may leave a single block of the grid
that it covers whole: a block accepted there names the tagging mode's grouped depth
expression, like any other.  Axis-aligned right triangles with their corner half a pixel
before every offset modulo 16, one per 64x64 cell; IDs, depth bits and classes are equal.
"""
import numpy as np
import pytest

from ifrit_hip import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu

W = H = 1024
EYE = np.eye(4, dtype=np.float32)


def _corners(z):
    k = np.arange(256)
    c = np.stack([k % 16, k // 16], -1)
    p = (c * 64 + c - 0.5)[:, None, :] + np.array([[0.0, 0.0], [45.0, 0.0], [0.0, 45.0]])
    clip = np.empty((256, 3, 4), np.float32)
    clip[..., :2] = p / W * 2 - 1
    clip[..., 2] = z + np.array([0.0, 0.07, 0.11])
    clip[..., 3] = 1.0
    idx = np.arange(768, dtype=np.int32).reshape(-1, 3)
    return clip.reshape(-1, 4), np.concatenate([idx, idx[:, ::-1]]).reshape(-1)


def _bind(r, clip, idx):
    r.set_target(W, H, 1)
    r.bind_geometry(clip, idx, EYE, clip_passthrough=True)
    r.bind_fragment_program(scenes.Scene("t", W, H, 1, clip, idx, EYE, program=scenes.PROGRAM_FLAT))


@pytest.mark.parametrize("tagging", [True, False])
def test_not_equal_cleared(renderer_factory, tagging):
    r = renderer_factory()
    r.set_deterministic(not tagging)
    r.set_depth_func(5)
    clip, idx = _corners(0.3)
    _bind(r, clip, idx)
    print(f"[ordered blocks NOT_EQUAL tagging={tagging}]", flush=True)
    r.draw()
    f = O.Frame().render(W, H, 1, clip, idx, depth_func=5, tagging=tagging)
    ids, depth = r.visibility()
    assert (f.ids != 0xFFFFFFFF).sum() > 200000 and ((f.cls == 4).any() or not tagging)
    assert np.array_equal(ids, f.ids)
    assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
    assert np.array_equal(r.coverage_class(), f.cls)


@pytest.mark.parametrize("tagging", [True, False])
@pytest.mark.parametrize("func", [2, 5, 3])
def test_second_pass_without_clear(renderer_factory, func, tagging):
    """LESS by the keys, then the same triangles again by the fold."""
    r = renderer_factory()
    r.set_deterministic(not tagging)
    clip, idx = _corners(0.3)
    _bind(r, clip, idx)
    r.draw()
    d0, c0 = r.visibility()[1], r.coverage_class()
    r.set_depth_func(func)
    print(f"[ordered blocks func={func} tagging={tagging} without clear]", flush=True)
    r.draw(clear=False)
    f = O.Frame().render(W, H, 1, clip, idx, depth_func=func, tagging=tagging, clear=False, depth_in=d0)
    ids, depth = r.visibility()
    won = f.ids != 0xFFFFFFFF
    assert won.sum() > 200000 or func == 5
    assert np.array_equal(ids[won], f.ids[won])
    assert np.array_equal(depth.view(np.uint32), f.depth.view(np.uint32))
    assert np.array_equal(r.coverage_class(), np.where(won, f.cls, c0))
