"""Colours of pixels that keep a record of an earlier, larger draw.

Draws without clear shade every pixel again, those they leave alone by the slot of
the draw that won them: 12k triangles and then two, or a few lines, over them (slots
beyond the second draw's records and beyond every clip fan it reserves, 4096 at the
least), and a textured scene followed by its own first triangles, of which none
passes; and a scissored draw of a few over 12k, which keeps slots outside its
rectangle.  A draw whose tile lists do not fit draws nothing and must leave the
colours alone.  Flat colours follow the primitive IDs (at most 16 roundings, as in the
shading-order tests); the textured frame must not change by a bit.
"""
import numpy as np
import pytest

from ifrit_hip import IfritError, scenes
from oracle import oracle as O

from test_gpu_shade_order import _flat, _scene

pytestmark = pytest.mark.gpu

EYE = np.eye(4, dtype=np.float32)
BLACK = np.zeros(4)


def _overlay():
    clip = np.array([[-0.9, -0.8, 0.05, 1], [0.7, -0.5, 0.05, 1], [-0.2, 0.9, 0.05, 1],
                     [0.9, 0.8, 0.04, 1], [-0.6, 0.7, 0.04, 1], [0.1, -0.9, 0.04, 1]], np.float32)
    return clip, np.array([0, 1, 2, 2, 1, 0, 3, 4, 5, 5, 4, 3], np.int32)


def _bind(r, W, H, samples, clip, idx):
    r.bind_geometry(clip, idx, EYE, clip_passthrough=True)
    r.bind_fragment_program(scenes.Scene("t", W, H, samples, clip, idx, EYE, program=scenes.PROGRAM_FLAT))


@pytest.mark.parametrize("samples", [1, 4])
def test_small_draw_over_a_large_one(renderer_factory, samples):
    r = renderer_factory()
    r.set_float_output(True)
    W, H = 320, 201
    clip, idx = _scene(np.random.default_rng(samples), W, H, 5600)
    over, oi = _overlay()
    f = O.Frame().render(W, H, samples, clip, idx)
    g = O.Frame().render(W, H, samples, over, oi, clear=False, depth_in=f.depth)
    r.set_target(W, H, samples)
    _bind(r, W, H, samples, clip, idx)
    r.draw()
    _bind(r, W, H, samples, over, oi)
    print(f"[kept slots s={samples}]", flush=True)
    r.draw(clear=False)
    ids = np.where(g.ids != 0xFFFFFFFF, g.ids, f.ids)
    assert (g.ids != 0xFFFFFFFF).any() and (f.ids[g.ids == 0xFFFFFFFF] > 5000).any()
    assert np.array_equal(r.visibility()[0], ids)
    want = _flat(ids.reshape(H, W, samples), BLACK).mean(2)
    assert np.abs(r.color_f32().reshape(H, W, 4) - want).max() < 1e-6


def test_lines_over_a_large_draw(renderer_factory):
    r = renderer_factory()
    r.set_float_output(True)
    W, H = 320, 201
    clip, idx = _scene(np.random.default_rng(7), W, H, 5600)
    clip[:36, 0] = 3.0  # the slots that the lines' records take hold no pixel
    over, oi = _overlay()
    f = O.Frame().render(W, H, 1, clip, idx)
    g = O.Frame().render_polygons(W, H, over, oi, 1, clear=False, depth_in=f.depth)
    r.set_target(W, H, 1)
    _bind(r, W, H, 1, clip, idx)
    r.draw()
    r.set_polygon_mode(1)
    _bind(r, W, H, 1, over, oi)
    print("[kept slots, lines]", flush=True)
    r.draw(clear=False)
    line = g.ids != 0xFFFFFFFF
    assert line.any() and (f.ids[~line & (f.ids != 0xFFFFFFFF)] > 5000).any()
    want = _flat(np.where(line, g.ids // 3, f.ids).reshape(H, W), BLACK)
    assert np.abs(r.color_f32().reshape(H, W, 4) - want).max() < 1e-6


@pytest.mark.parametrize("samples", [1, 4])
def test_first_triangles_of_a_textured_scene(renderer_factory, samples):
    s = scenes.config2(200, 150, samples, spheres=8, tex_size=64)
    assert s.num_triangles == 40960
    r = renderer_factory()
    r.set_float_output(True)
    r.load_scene(s)
    assert r.draw()["clippedTriangles"] == 0
    before = r.color_f32()
    r.num_indices = 6
    print(f"[kept slots, textured s={samples}]", flush=True)
    st = r.draw(clear=False)
    assert st["inputTriangles"] == 2
    assert np.array_equal(r.color_f32().view(np.uint32), before.view(np.uint32))


@pytest.mark.parametrize("samples", [1, 8])
@pytest.mark.parametrize("tile", [8, 32])
def test_scissored_small_draw_over_a_large_one(renderer_factory, tile, samples):
    s = scenes.config2(200, 150, samples, spheres=8, tex_size=64)
    r = renderer_factory()
    r.set_tuning(shadeTile=tile)
    r.set_float_output(True)
    r.load_scene(s)
    r.draw()
    before = r.color_f32()
    r.set_clear_values((0.25, 0.5, 0.75, 1.0))
    r.num_indices = 3 * 2 * 5120  # the first two spheres, one inside the scissor
    r.draw()
    alone = r.color_f32()
    r.set_clear_values()
    r.num_indices = s.indices.size
    r.draw()
    r.set_clear_values((0.25, 0.5, 0.75, 1.0))
    r.set_scissors([(21.0, 18.0, 102.0, 90.0)])
    r.num_indices = 3 * 2 * 5120
    print(f"[kept slots, scissor s={samples} tile={tile}]", flush=True)
    r.draw()
    y, x = np.mgrid[:s.height, :s.width]
    inside = ((x >= 21) & (x <= 123) & (y >= 18) & (y <= 108))[..., None]
    assert np.array_equal(r.color_f32(), np.where(inside, alone, before))


@pytest.mark.parametrize("part", [256, 512])
@pytest.mark.parametrize("clear", [True, False])
def test_overflowing_draw_shades_nothing(renderer_factory, clear, part):
    r = renderer_factory()
    r.set_tuning(rasterPartEntries=part)
    W, H = 320, 201
    small, si = _overlay()
    large, li = _scene(np.random.default_rng(3), W, H, 5600)
    r.set_target(W, H, 4)
    _bind(r, W, H, 4, large, li)
    r.draw()
    want = r.color()
    _bind(r, W, H, 4, small, si)
    r.draw()
    before = r.color()
    _bind(r, W, H, 4, large, li)
    r.set_tuning(binCapacity=4096)
    print(f"[kept slots, overflow clear={clear} part={part}]", flush=True)
    r.draw_async(clear=clear)
    with pytest.raises(IfritError, match="binning buffers"):
        r.synchronize()
    assert np.array_equal(r.color(), before)
    r.draw()  # the buffers have grown
    assert np.array_equal(r.color(), want)


@pytest.mark.parametrize("mode", [0, 1])
def test_cull_mode_with_swap_flags_after_a_large_draw(renderer_factory, mode):
    s = scenes.config2(200, 150, 1, spheres=8, tex_size=64)
    r = renderer_factory()
    r.set_float_output(True)
    r.load_scene(s)
    r.draw()
    before = r.color_f32()
    r.set_cull_mode(mode)
    r.num_indices = 6
    print(f"[kept slots, cull mode {mode}]", flush=True)
    r.draw(clear=False)  # behind the sphere's front
    assert np.array_equal(r.color_f32().view(np.uint32), before.view(np.uint32))


@pytest.mark.parametrize("samples", [1, 4])
def test_clip_fans_of_a_large_draw(renderer_factory, samples):
    """The ground crosses w = 0: its pixels keep fans, whose weights the next draw must not lose."""
    s = scenes.config1(200, 150)
    s.samples = samples
    r = renderer_factory()
    r.set_float_output(True)
    r.load_scene(s)
    assert r.draw()["clippedTriangles"] > 0
    assert (r.visibility()[0] == s.num_triangles - 1).sum() > 1000
    before = r.color_f32()
    r.num_indices = 6
    print(f"[kept slots, fans s={samples}]", flush=True)
    assert r.draw(clear=False)["clippedTriangles"] == 0
    assert np.array_equal(r.color_f32().view(np.uint32), before.view(np.uint32))


@pytest.mark.parametrize("large", ["meshlets", "short records"])
def test_small_buffers_after_a_large_draw(renderer_factory, large):
    """Kept triangles and vertices beyond the second draw's buffers: their colour is of no use, but
    the second draw's own pixels are as when it draws alone."""
    s = scenes.config2(200, 150, 1, spheres=8, tex_size=64)
    clip, oi = _overlay()
    over = np.random.default_rng(1).uniform(0.1, 0.9, (6, 8 if large == "meshlets" else 256)).astype(np.float32)
    over[:, :4] = clip
    small = scenes.Scene("t", 200, 150, 1, over, oi, EYE, program=s.program, sampler=s.sampler, lights=s.lights,
                         textures=s.textures)
    r = renderer_factory()
    r.set_float_output(True)
    if large == "meshlets":
        recs, loc, vo, io, _ = scenes.build_meshlets(s.vertices, s.indices)
        r.set_target(200, 150, 1)
        for t in s.textures:
            r.add_texture(t)
        r.bind_fragment_program(small)
        for slot, a in enumerate((recs, loc, vo, io)):
            r.create_buffer(slot, a)
        r.bind_meshlets(s.mvp, recs.shape[1])
        r.bind_geometry(over, oi, EYE, clip_passthrough=True)
        r.draw_mesh_tasks(len(vo) - 1)
    else:
        r.load_scene(s)
        r.draw()
        r.bind_geometry(over, oi, EYE, clip_passthrough=True)
        r.bind_fragment_program(small)
    assert (r.visibility()[0] != 0xFFFFFFFF).sum() > 1000
    print(f"[kept slots, small buffers after {large}]", flush=True)
    r.draw(clear=False)
    got = r.color_f32().reshape(-1, 4)
    r.draw()
    own = r.visibility()[0] != 0xFFFFFFFF
    assert 1000 < own.sum() < own.size
    assert np.array_equal(got[own].view(np.uint32), r.color_f32().reshape(-1, 4)[own].view(np.uint32))


@pytest.mark.parametrize("samples", [1, 4, 8])
def test_pixels_no_draw_has_written(renderer_factory, samples):
    """The first draw of a renderer, and one into a larger target, under a scissor."""
    r = renderer_factory()
    clip, idx = _overlay()
    for W, H in [(64, 33), (321, 200)]:
        r.set_target(W, H, samples)
        _bind(r, W, H, samples, clip, idx)
        r.set_scissors([(5.0, 3.0, 31.0, 20.0)])
        print(f"[no draw yet s={samples} {W}x{H}]", flush=True)
        r.draw()
        f = O.Frame().render(W, H, samples, clip, idx)
        y, x = np.mgrid[:H, :W]
        inside = np.repeat(((x >= 5) & (x <= 36) & (y >= 3) & (y <= 23)).reshape(-1), samples)
        ids = r.visibility()[0]
        assert (ids[~inside] == 0xFFFFFFFF).all()
        assert np.array_equal(ids[inside], f.ids[inside])


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("n", [1, 63, 130, 1365])
def test_same_fans_keep_their_slots(renderer_factory, n, samples):
    """n triangles across w = 0 among as many others, drawn again without clear: nothing passes, and
    primitive IDs and colours must not change (1365: as many as the smallest capacity ranks)."""
    rng = np.random.default_rng(n)
    W, H = 200, 150
    xyz = np.concatenate([rng.uniform(-1, 1, (2 * n, 3, 2)), rng.uniform(0.2, 0.8, (2 * n, 3, 1))], -1)
    w = rng.uniform(0.5, 2.0, (2 * n, 3, 1))
    w[::2, 0] *= -1.0  # one corner of every other one behind the eye
    v = np.concatenate([xyz * np.abs(w), w, rng.uniform(-1, 1, (2 * n, 3, 8))], -1).reshape(-1, 12).astype(np.float32)
    i = np.arange(6 * n, dtype=np.int32).reshape(-1, 3)
    idx = np.ascontiguousarray(np.where(rng.random((2 * n, 1)) < 0.5, i, i[:, ::-1])).reshape(-1)
    r = renderer_factory()
    r.set_float_output(True)
    r.set_cull_mode(0)
    r.set_target(W, H, samples)
    r.bind_geometry(v, idx, EYE, clip_passthrough=True)
    r.bind_fragment_program(scenes.Scene("t", W, H, samples, v, idx, EYE, program=scenes.PROGRAM_NORMAL_LAMBERT,
                                         lights=[((0.3, 0.5, 0.8, 0.0), (1.0, 0.9, 0.8, 0.0))]))
    assert r.draw()["clippedTriangles"] >= n
    ids, color = r.visibility()[0], r.color_f32()
    for k in range(3):
        print(f"[kept slots, same fans n={n} s={samples} {k}]", flush=True)
        r.draw(clear=False)
        assert np.array_equal(r.visibility()[0], ids)
        assert np.array_equal(r.color_f32().view(np.uint32), color.view(np.uint32))
