"""What the renderer's speed is measured on: whole draws through its public
entry points, from the smallest off-screen query to the 8x MSAA frame, the
multi-view batch and the two materials.

Three ways a program calls the library, each with its own kinds of case:

* ``device``: the caller holds vertices and indices in device memory and wants
  primitive IDs, depth and colour there (iftrDrawNoAlloc with torch tensors);
* ``frame``: the renderer holds the scene, the program draws a frame and takes
  the image to host memory (iftrDrawLegacy, then the RGBA8 or FP32 colour into
  a pinned buffer that it keeps from frame to frame);
* ``views``: one draw of many cameras as a replayed graph, every shaded view's
  colour and every depth-only view's depth taken to host memory.

Scenes are the repository's seeded generators (ifrit_hip.scenes); the seed
places the spheres, turns them and draws their textures, or raises the height
field, and moves the camera of the fixed scenes.
"""
import ctypes as C
import dataclasses
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ifrit-v2_amd"))

import ifrit_hip  # noqa: E402
from ifrit_hip import Renderer, scenes  # noqa: E402

# IfritBlendFactor names: the factor named SRC_ALPHA weighs by 1 - source alpha, as in the reference
BLEND_ONE, BLEND_SRC_ALPHA, BLEND_ONE_MINUS_SRC_ALPHA = 1, 6, 7
LESS, LESS_OR_EQUAL = 1, 3
TRIS = {2: 320, 3: 1280, 4: 5120}     # triangles of an icosphere by subdivision level
VERTS = {2: 162, 3: 642, 4: 2562}


def listed():
    return [
        # an occlusion or picking query: one small object, IDs and depth only; latency is all
        dict(name="device_query_256", kind="device", scene="sphere", width=256, height=256, samples=1, shade=False),
        # a preview or a thumbnail in a service that keeps its meshes on the device: 4x MSAA at an odd size
        dict(name="device_1009x767_4x", kind="device", scene="spheres", width=1009, height=767, samples=4, spheres=12,
             level=4, tex=512, shade=True),
        # a full-HD frame of a moderate scene, 16x anisotropic Blinn-Phong, everything on the device
        dict(name="device_1080p", kind="device", scene="spheres", width=1920, height=1080, samples=1, spheres=25,
             level=4, tex=1024, shade=True),
        # the small classic frame: a few thousand triangles, one of them across w = 0, trilinear checker
        dict(name="frame_640x480", kind="frame", scene="config1", width=640, height=480, samples=1),
        # the headline frame: 1.3M triangles, 8x MSAA, 256 textures of 2048 texels a side
        dict(name="frame_1080p_8x", kind="frame", scene="spheres", width=1920, height=1080, samples=8, spheres=256,
             level=4, tex=2048),
        # terrain: 4.2M triangles of about half a pixel below 16 screen-sized ones, flat colour, 4x MSAA
        dict(name="frame_1080p_4x_terrain", kind="frame", scene="heightfield", width=1920, height=1080, samples=4,
             cells=2048, big=16),
        # the CPU path's own workload: FP32 colour, one sample, normal-Lambert
        dict(name="frame_720p_fp32", kind="frame", scene="lambert", width=1280, height=720, samples=1, spheres=256,
             level=4),
        # translucent objects, blended in primitive order
        dict(name="frame_720p_blend", kind="frame", scene="translucent", width=1280, height=720, samples=1,
             spheres=64, level=3),
        # a depth function other than LESS (a later pass over an equal depth), which folds fragments in order
        dict(name="frame_720p_4x_lequal", kind="frame", scene="spheres", width=1280, height=720, samples=4,
             spheres=64, level=3, tex=512, depth_func=LESS_OR_EQUAL),
        # the layered material and the network that replaces it
        dict(name="frame_1080p_ggx", kind="frame", scene="ggx", width=1920, height=1080, samples=1, spheres=256,
             level=4, tex=2048),
        dict(name="frame_1080p_neural", kind="frame", scene="neural", width=1920, height=1080, samples=1, spheres=256,
             level=4, tex=2048),
        # a batch of shadow cascades, cube faces (triangles across w = 0) and shaded cameras of uneven size
        dict(name="views_34", kind="views", scene="spheres", spheres=256, level=4, tex=1024, cascades=4,
             cascade_size=1024, cube_size=512, cameras=24, max_width=640, max_height=480),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds: sizes over their whole range, odd ones included."""
    pick = rng.choice(["query", "device", "device", "config1", "spheres", "spheres", "heightfield", "lambert",
                       "translucent", "lequal", "ggx", "neural", "views"])
    if pick == "query":
        return dict(kind="device", scene="sphere", width=_log(rng, 64, 640), height=_log(rng, 64, 480), samples=1,
                    shade=False)
    if pick == "device":
        s = rng.choice([1, 1, 4, 8])
        # the entry point's scratch holds 1920x1080 at one sample with 128K triangles, or 1024x1024 at four with 64K
        px = {1: 1920 * 1080, 4: 1024 * 800, 8: 512 * 800}[s]
        w = _log(rng, 160, 1920 if s == 1 else 1100)
        return dict(kind="device", scene="spheres", width=w, height=max(16, min(1080, _log(rng, 120, 1080), px // w)),
                    samples=s, spheres=rng.randint(1, {1: 25, 4: 12, 8: 10}[s]), level=rng.choice([3, 4]),
                    tex=rng.choice([256, 512, 1024]), shade=rng.random() < 0.7)
    w, h = _log(rng, 192, 1920), _log(rng, 160, 1080)
    if pick == "config1":
        return dict(kind="frame", scene="config1", width=w, height=h, samples=1)
    if pick == "spheres":
        return dict(kind="frame", scene="spheres", width=w, height=h, samples=rng.choice([1, 4, 8, 8]),
                    spheres=_log(rng, 4, 256), level=rng.choice([3, 4, 4]), tex=rng.choice([512, 1024]))
    if pick == "heightfield":
        return dict(kind="frame", scene="heightfield", width=w, height=h, samples=rng.choice([1, 4, 8]),
                    cells=_log(rng, 128, 2048) // 2 * 2, big=rng.randint(0, 16))
    if pick == "lambert":
        return dict(kind="frame", scene="lambert", width=min(w, 1280), height=min(h, 720), samples=1,
                    spheres=_log(rng, 4, 256), level=4)
    if pick == "translucent":
        return dict(kind="frame", scene="translucent", width=min(w, 1280), height=min(h, 720), samples=1,
                    spheres=rng.randint(4, 64), level=rng.choice([2, 3]))
    if pick == "lequal":
        return dict(kind="frame", scene="spheres", width=min(w, 1280), height=min(h, 720), samples=rng.choice([1, 4]),
                    spheres=rng.randint(4, 64), level=rng.choice([2, 3]), tex=512,
                    depth_func=rng.choice([LESS_OR_EQUAL, 6, 7]))
    if pick in ("ggx", "neural"):
        return dict(kind="frame", scene=pick, width=w, height=h, samples=1, spheres=_log(rng, 8, 256), level=4,
                    tex=rng.choice([512, 1024]))
    return dict(kind="views", scene="spheres", spheres=_log(rng, 8, 256), level=rng.choice([3, 4]), tex=512,
                cascades=rng.randint(1, 4), cascade_size=rng.choice([333, 512, 1024]), cube_size=rng.choice([129, 256, 512]),
                cameras=rng.randint(1, 24), max_width=rng.choice([320, 511, 640]), max_height=rng.choice([270, 480]))


# ---------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------

def _scene(case, seed):
    kind, w, h = case["scene"], case.get("width", 64), case.get("height", 64)
    if kind in ("config1", "sphere"):
        s = scenes.config1(w, h)
        rng = np.random.default_rng(seed)
        eye = (0.6 + float(rng.uniform(-0.4, 0.4)), 1.2 + float(rng.uniform(-0.3, 0.3)), -3.2)
        mvp = (scenes.perspective(math.radians(60.0), w / h, 0.1, 100.0) @ scenes.look_at(eye, (0, 0, 0), (0, 1, 0)))
        s = dataclasses.replace(s, mvp=mvp.astype(np.float32), camera=eye)
        if kind == "sphere":  # without the ground
            s = dataclasses.replace(s, vertices=s.vertices[:-4], indices=s.indices[:-6])
        return s
    if kind == "heightfield":
        return scenes.config3(w, h, case["samples"], gx=case["cells"], gy=case["cells"] // 2, big=case["big"],
                              seed=seed % (1 << 20))
    if kind == "lambert":
        return scenes.normal_lambert(scenes.config2(w, h, 1, case["spheres"], case["level"], 16, seed=seed))
    if kind in ("ggx", "neural"):
        # the layers' texels come from the device generator: what the layers hold does not change the work
        s = scenes.config5(w, h, 1, case["spheres"], case["level"], 16, seed=seed)
        t, lv = case["tex"], scenes.num_levels(case["tex"], case["tex"])
        return dataclasses.replace(s, textures=[scenes.Texture(t, t, lv, None, (seed + k) & 0x7FFFFFFF)
                                                for k in range(3)])
    s = scenes.config2(w, h, case.get("samples", 1), case["spheres"], case["level"], case.get("tex", 16), seed=seed)
    if kind == "translucent":
        s = dataclasses.replace(s, program=scenes.PROGRAM_FLAT_ALPHA, textures=[])
    return s


def _views(case, seed):
    """The seed's cameras; the sizes of the shaded views are the case's own, uneven."""
    views = scenes.config4_views(seed, case["cascades"], case["cascade_size"], 6, case["cube_size"], case["cameras"],
                                 (case["max_width"], case["max_height"]), 192)
    rng = np.random.default_rng(case["cameras"])
    for v in views:
        if v["shade"]:
            w, h = int(rng.integers(192, case["max_width"] + 1)), int(rng.integers(192, case["max_height"] + 1))
            m = v["mvp"].astype(np.float64)
            m[0] *= (v["width"] / v["height"]) / (w / h)  # the same vertical field of view at the new aspect
            v.update(width=w, height=h, mvp=m.astype(np.float32))
    return views


def _params(seed):
    """Xavier-uniform network weights in the library's layout (W1[16][64], b1, W2[64][64], b2, W3[64][4], b3)."""
    rng = np.random.default_rng(seed)
    p = np.zeros(ifrit_hip.NEURAL_PARAMS, np.float32)
    p[0:1024].reshape(16, 64)[:14] = rng.uniform(-1, 1, (14, 64)) * math.sqrt(6 / 78)
    p[1024:1088] = rng.uniform(-0.1, 0.1, 64)
    p[1088:5184] = (rng.uniform(-1, 1, (64, 64)) * math.sqrt(6 / 128)).reshape(-1)
    p[5184:5248] = rng.uniform(-0.1, 0.1, 64)
    p[5248:5504].reshape(64, 4)[:, :3] = rng.uniform(-1, 1, (64, 3)) * math.sqrt(6 / 67)
    p[5504:5507] = rng.uniform(0.2, 0.6, 3)
    return p


class _State:
    """A renderer with its scene, and the buffers the program reads frames into."""


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def prepare(case, seed):
    st = _State()
    st.kind = case["kind"]
    s = _scene(case, seed)
    r = st.r = Renderer()
    r.load_scene(s)
    r.set_clear_values((0.0, 0.0, 0.0, 0.0), 1.0)  # depth cleared to the far plane
    h, w, spp = s.height, s.width, s.samples
    if st.kind == "device":
        st.vtx = torch.from_numpy(np.ascontiguousarray(s.vertices)).cuda()
        st.idx = torch.from_numpy(np.ascontiguousarray(s.indices)).cuda()
        st.ids = torch.empty((h, w, spp), dtype=torch.int32, device="cuda")
        st.depth = torch.empty((h, w, spp), dtype=torch.float32, device="cuda")
        st.rgba = torch.empty((h, w, 4), dtype=torch.uint8, device="cuda") if case["shade"] else None
        st.desc = ifrit_hip.NoAllocDraw(_ptr(st.vtx), st.vtx.shape[1], st.vtx.shape[0], _ptr(st.idx),
                                        st.idx.numel(), _ptr(st.ids), _ptr(st.depth),
                                        _ptr(st.rgba) if case["shade"] else None)
        torch.cuda.synchronize()
        return st
    if st.kind == "views":
        views = _views(case, seed)
        r.set_views(views)
        r.set_graph_mode(True)
        st.out = [torch.empty((v["height"], v["width"], 4), dtype=torch.uint8, pin_memory=True) if v["shade"] else
                  torch.empty((v["height"], v["width"]), dtype=torch.float32, pin_memory=True) for v in views]
        return st
    st.fp32 = case["scene"] == "lambert"
    if case["scene"] == "neural":
        # one step at learning rate 0 lays out the latent texture; the weights are the seed's
        r.train_neural(views=4, view_size=(128, 128), max_fragments=1 << 16, steps=1, batch=256, lr_latent=0.0,
                       lr_mlp=0.0, seed=seed & 0x7FFFFFFF, latent_size=min(1024, case["tex"]), single_tap=True)
        r.set_neural_params(_params(seed))
        r.bind_fragment_program(s, program=4, precision=0)
    if case["scene"] == "translucent":
        r.set_blend((BLEND_ONE_MINUS_SRC_ALPHA, BLEND_SRC_ALPHA, BLEND_ONE, BLEND_SRC_ALPHA))
    if "depth_func" in case:
        r.set_depth_func(case["depth_func"])
    if st.fp32:
        r.set_float_output(True)
    st.out = torch.empty((h, w, 4), dtype=torch.float32 if st.fp32 else torch.uint8, pin_memory=True)
    return st


def run(st):
    r = st.r
    if st.kind == "device":
        r.L.iftrDrawNoAlloc(r.h, C.byref(st.desc))
        r._check()
        return {"ids": st.ids, "depth": st.depth, "rgba": st.rgba}
    r.draw()
    if st.kind == "views":
        for v, out in enumerate(st.out):
            if out.dtype == torch.uint8:
                r.L.iftrGetViewColorRGBA8(r.h, v, _ptr(out))
            else:
                r.L.iftrGetViewVisibility(r.h, v, None, _ptr(out))
        r._check()
        return st.out
    if st.fp32:
        r.L.iftrGetColorRGBA32F(r.h, _ptr(st.out))
    else:
        r.L.iftrGetColorRGBA8(r.h, _ptr(st.out))
    r._check()
    return st.out


def work(case):
    """Vertices and indices read once, outputs written once, one texel with its mip chain per shaded pixel (the
    share of the frame the scene covers: about a third for the spheres).  Operations: the transform of every
    vertex, the edges of every front-facing triangle, the lighting of covered pixels, the network's multiplies."""
    kind = case["scene"]
    if kind in ("config1", "sphere"):
        V, T, stride = 65 * 33 + 4, 4098, 8
    elif kind == "heightfield":
        n = case["cells"]
        V, T, stride = (n + 1) * (n // 2 + 1) + 3 * case["big"], n * (n // 2) * 2 + case["big"], 3
    else:
        V, T = VERTS[case["level"]] * case["spheres"], TRIS[case["level"]] * case["spheres"]
        stride = 11 if kind in ("ggx", "neural") else 8
    inputs = V * stride * 4 + T * 12
    if case["kind"] == "views":
        deep = case["cascades"] * case["cascade_size"] ** 2 + 6 * case["cube_size"] ** 2
        shaded = case["cameras"] * ((192 + case["max_width"]) // 2) * ((192 + case["max_height"]) // 2)
        n = case["cascades"] + 6 + case["cameras"]
        return {"bytes": inputs + deep * 4 + shaded * (4 + 4 * 4 / 9), "flops": n * (V * 28 + T * 50) + shaded * 100}
    px = case["width"] * case["height"]
    flops = V * 28 + T * 50
    if case["kind"] == "device":
        out = px * case["samples"] * 8 + (px * (4 + 4 * 4 / 9) if case["shade"] else 0)
        return {"bytes": inputs + out, "flops": flops + (px * 100 if case["shade"] else 0)}
    out = px * (16 if kind == "lambert" else 4)
    if kind in ("spheres", "config1"):
        out += px * 4 * 4 / 9
    elif kind == "ggx":
        out += px * 3 * 4 * 4 / 9
    elif kind == "neural":
        out += px * 16 * 4 / 9
        flops += px / 3 * 10368
    return {"bytes": inputs + out, "flops": flops + px * 35}


# ---------------------------------------------------------------------------
# the same images in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _raster64(vertices, indices, mvp, w, h):
    """Nearest front-facing triangle at every pixel's corner, in 64 bits: its depth (1 where there is none), its
    index and its screen-space weights.  For triangles with w > 0 throughout."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    v = torch.from_numpy(np.ascontiguousarray(vertices[:, :3])).to(dev, torch.float64)
    m = torch.from_numpy(np.ascontiguousarray(mvp)).to(dev, torch.float64)
    c = torch.cat([v, torch.ones_like(v[:, :1])], 1) @ m.T
    t = torch.from_numpy(np.ascontiguousarray(indices)).to(dev, torch.int64).reshape(-1, 3)
    sx, sy = (c[:, 0] / c[:, 3] + 1) * (0.5 * w), (c[:, 1] / c[:, 3] + 1) * (0.5 * h)
    sz = c[:, 2] / c[:, 3]
    X, Y, Z, wc = sx[t], sy[t], sz[t], c[:, 3][t]
    area = (X[:, 1] - X[:, 0]) * (Y[:, 2] - Y[:, 0]) - (X[:, 2] - X[:, 0]) * (Y[:, 1] - Y[:, 0])
    x0, x1 = X.amin(1).ceil().clamp(0, w), X.amax(1).floor().clamp(-1, w - 1)
    y0, y1 = Y.amin(1).ceil().clamp(0, h), Y.amax(1).floor().clamp(-1, h - 1)
    seen = (area > 0) & (x1 >= x0) & (y1 >= y0) & (wc.amin(1) > 0) & (Z.amax(1) >= 0) & (Z.amin(1) <= 1)
    tri = seen.nonzero()[:, 0]
    bw = (x1 - x0 + 1)[tri].to(torch.int64)
    n = bw * (y1 - y0 + 1)[tri].to(torch.int64)
    depth = torch.ones(w * h, dtype=torch.float64, device=dev)
    best = torch.full((w * h,), -1, dtype=torch.int64, device=dev)
    lam = torch.zeros(w * h, 3, dtype=torch.float64, device=dev)
    ends = n.cumsum(0)
    for part in (1, 2):  # the least depth first, then the triangle that has it
        a = 0
        while a < tri.numel():
            base = int(ends[a - 1]) if a else 0
            b = max(a + 1, int(torch.searchsorted(ends, base + 20_000_000, right=True)))
            k = torch.repeat_interleave(torch.arange(a, b, device=dev), n[a:b])
            off = torch.arange(k.numel(), device=dev) - (ends[a:b] - n[a:b] - base)[k - a]
            q = tri[k]
            px, py = x0[q] + off % bw[k], y0[q] + off // bw[k]
            l0 = ((X[q, 2] - X[q, 1]) * (py - Y[q, 1]) - (Y[q, 2] - Y[q, 1]) * (px - X[q, 1])) / area[q]
            l1 = ((X[q, 0] - X[q, 2]) * (py - Y[q, 2]) - (Y[q, 0] - Y[q, 2]) * (px - X[q, 2])) / area[q]
            l2 = 1 - l0 - l1
            z = l0 * Z[q, 0] + l1 * Z[q, 1] + l2 * Z[q, 2]
            pix = py.to(torch.int64) * w + px.to(torch.int64)
            ok = (l0 >= 0) & (l1 >= 0) & (l2 >= 0)
            if part == 1:
                depth.scatter_reduce_(0, pix[ok], z[ok], "amin")
            else:
                ok &= (z == depth[pix]) & (z < 1)
                best[pix[ok]] = q[ok]
                lam[pix[ok]] = torch.stack([l0, l1, l2], 1)[ok] / wc[q[ok]]
            a = b
    return depth, best, lam / lam.sum(1, keepdim=True).clamp(min=1e-300), t


def exact(case, seed):
    """Depth of the one-sample draws without triangles across w = 0, and the normal-Lambert colour; the other
    outputs are IDs and RGBA8."""
    if case["kind"] == "device" and case["samples"] == 1:
        s = _scene(case, seed)
        depth = _raster64(s.vertices, s.indices, s.mvp, s.width, s.height)[0]
        return {"ids": None, "depth": depth.reshape(s.height, s.width, 1).cpu(), "rgba": None}
    if case["kind"] == "views":
        s, out = _scene(case, seed), []
        for v in _views(case, seed):
            if v["kind"] == "cascade":
                d = _raster64(s.vertices, s.indices, v["mvp"], v["width"], v["height"])[0]
                out.append(d.reshape(v["height"], v["width"]).cpu())
            else:
                out.append(None)
        return out
    if case["scene"] == "lambert":
        s = _scene(case, seed)
        _, best, lam, t = _raster64(s.vertices, s.indices, s.mvp, s.width, s.height)
        nrm = torch.from_numpy(np.ascontiguousarray(s.vertices[:, 3:6])).to(best.device, torch.float64)
        N = (nrm[t[best.clamp(min=0)]] * lam[:, :, None]).sum(1)
        light = torch.tensor(s.lights[0][0][:3], dtype=torch.float64, device=best.device)
        d = ((N @ light) / (N.norm(dim=1) ** 2 + 1e-20).sqrt()).clamp(min=0)
        rgb = s.ambient + torch.tensor(s.lights[0][1][:3], dtype=torch.float64, device=best.device) * d[:, None] \
            + (d ** s.shininess)[:, None]
        out = torch.cat([rgb.clamp(0, 1), torch.ones_like(rgb[:, :1])], 1) * (best >= 0)[:, None]
        return out.reshape(s.height, s.width, 4).cpu()
    return None
