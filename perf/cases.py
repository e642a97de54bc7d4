"""The work this renderer is used for, as cases that can be timed and compared.

A case is a plain dict.  `listed()` names the fixed ones, `draw(rng)` makes more over the same
ranges, `prepare(case, seed)` builds what a program has in hand before the call (device buffers,
a Rasterizer with its state, a Batch, a DiffRenderer), `run(state)` is one pass through the
public entry points and returns every buffer it fills, `work(case)` what a pass cannot do
without, and `exact(case, seed)` the outputs in 64 bits where they are rounded numbers.

Frames (colour and depth images, hashes) have no value in 64 bits: the draw contract fixes
every fp32 rounding of the reference's incremental chains, so their images are equal bit for
bit or wrong.  The differentiable renderer's image and gradients are rounded values of an
analytic formula; `exact` evaluates that formula in plain torch in fp64 (coverage and the
discrete silhouette choices in fp32, as the formula defines them).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from softwarerenderer_amd import api, diff, scenes

SPAN, BLOCK, ADAPTIVE = api.RasterMode.Span, api.RasterMode.Block, api.RasterMode.Adaptive
NONE, CCW, CW = api.CullMode.None_, api.CullMode.CCW, api.CullMode.CW


# ---- the cases ---------------------------------------------------------------------------


def frame(scene, program, tris, width, height, mode, cull=CW, tuned=False, sync=False,
          host=False, **more):
    return dict(kind="frame", scene=scene, program=program, tris=tris, width=width,
                height=height, mode=mode, cull=cull, tuned=tuned, sync=sync, host=host, **more)


def listed():
    return [
        # one triangle drawn synchronously, as the reference's VertexProcessorTest does: the
        # cost of a call
        frame("triangle", "rgb", 1, 640, 480, SPAN, NONE, sync=True, name="triangle"),
        # a small animated mesh at VGA, enqueued frame after frame
        frame("sphere", "depth", 16128, 640, 480, SPAN, name="sphere_vga"),
        # the scene of the reference's Benchmark program: large overlapping triangles
        frame("overdraw", "rgb", 40960, 640, 480, SPAN, NONE, name="overdraw"),
        # the dense full-HD frame, at the launch shape the autotuner picks for it
        frame("soup", "depth", 1_000_000, 1920, 1080, BLOCK, tuned=True, name="soup_hd"),
        # a mid-sized frame of ragged size with the built-in launch shape, both traversals
        frame("soup", "depth", 150_001, 1003, 701, ADAPTIVE, NONE, name="soup_ragged"),
        # clip-heavy geometry under a program that observes every fragment
        frame("clip", "hash", 30_000, 800, 600, BLOCK, NONE, name="clip_hash"),
        # the Box demo's textured shader over a full screen
        dict(kind="texture", scene="floor", tris=2, width=1280, height=720, texels=512, aniso=8,
             mode=SPAN, name="texture_floor"),
        # a depth-tested wireframe
        dict(kind="lines", scene="wire", draw="line", count=48384, width=1280, height=720,
             name="wireframe"),
        # many scenes of all sizes in one pass
        dict(kind="batch", scenes=48, lo=1000, hi=60_000, name="batch"),
        # fitting one view of a mesh with autograd: launches and host work count
        dict(kind="diff", subdiv=5, views=1, size=256, channels=3, api="autograd",
             name="diff_one_view"),
        # the multi-view optimisation step
        dict(kind="diff", subdiv=6, views=64, size=512, channels=3, api="l2",
             name="diff_64_views"),
        # several terrains at once, each with views of its own
        dict(kind="terrain", scenes=8, lo=64, hi=512, views=2, size=768, name="diff_terrain"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["texture", "lines", "lines", "batch", "diff", "diff",
                                       "terrain"])
    if kind == "frame":
        scene = rng.choice(["soup", "soup", "sphere", "sphere", "overdraw", "clip", "triangle"])
        w, h = _log(rng, 65, 1920), _log(rng, 65, 1080)
        mode, cull = rng.choice([SPAN, BLOCK, ADAPTIVE]), rng.choice([NONE, CCW, CW])
        hi = {"soup": 1_000_000, "sphere": 200_000, "overdraw": 40_960, "clip": 100_000,
              "triangle": 1}[scene]
        tris = 1 if hi == 1 else _log(rng, 50, hi)
        if scene == "overdraw":  # every triangle covers a good part of the screen
            w, h = min(w, 800), min(h, 600)
        program = rng.choice({"soup": ["depth", "depth", "visibility", "hash", "coverage"],
                              "sphere": ["depth", "depth", "visibility", "hash"],
                              "overdraw": ["rgb"], "clip": ["depth", "hash"],
                              "triangle": ["rgb"]}[scene])
        host = tris < 100_000 and rng.random() < 0.12  # a program with buffers in host memory
        return frame(scene, program, tris, w, h, mode, cull, tuned=rng.random() < 0.3,
                     sync=host or scene == "triangle" or rng.random() < 0.3, host=host)
    if kind == "texture":
        return dict(kind=kind, scene=rng.choice(["floor", "sphere"]), tris=_log(rng, 100, 50_000),
                    width=_log(rng, 65, 1920), height=_log(rng, 65, 1080),
                    texels=rng.choice([64, 300, 512, 1024]), aniso=rng.choice([1, 4, 8, 16]),
                    mode=rng.choice([SPAN, BLOCK]))
    if kind == "lines":
        return dict(kind=kind, scene=rng.choice(["wire", "list", "list"]),
                    draw=rng.choice(["line", "line", "point"]), count=_log(rng, 30, 60_000),
                    width=_log(rng, 65, 1920), height=_log(rng, 65, 1080))
    if kind == "batch":
        return dict(kind=kind, scenes=_log(rng, 2, 64), lo=200, hi=_log(rng, 2_000, 60_000))
    if kind == "diff":
        views = _log(rng, 1, 32)
        return dict(kind=kind, subdiv=rng.randint(2, 6), views=views,
                    size=_log(rng, 50, 512 if views < 16 else 300),
                    channels=rng.choice([1, 3, 3, 4]), api=rng.choice(["autograd", "l2"]))
    return dict(kind=kind, scenes=rng.randint(2, 8), lo=24, hi=_log(rng, 64, 400),
                views=rng.randint(1, 3), size=_log(rng, 100, 700))


# ---- inputs ------------------------------------------------------------------------------


def _rings(tris):
    """Stacks of the UV sphere (slices = 2 stacks) of about `tris` triangles."""
    return max(3, int(round((1.0 + math.sqrt(1.0 + tris)) / 2.0)))


def _sphere(case, seed):
    n = _rings(case["tris"])
    return scenes.sphere_scene(n, 2 * n, seed=seed, width=case["width"], height=case["height"],
                               radius=np.random.default_rng(seed).uniform(0.85, 1.15))


def _scene(case, seed):
    w, h, t = case["width"], case["height"], case["tris"]
    if case["scene"] == "soup":
        return scenes.soup_scene(t, seed=seed, width=w, height=h)
    if case["scene"] == "sphere":
        return _sphere(case, seed)
    if case["scene"] == "clip":
        return scenes.clip_scene(t, seed=seed, width=w, height=h)
    rng = np.random.default_rng(seed)
    if case["scene"] == "overdraw":  # the distribution of Benchmark.cpp:66-105
        return scenes.Scene(rng.random((3 * t, 6), dtype=np.float32),
                            np.arange(3 * t, dtype=np.int32), np.eye(4, dtype=np.float32), w, h)
    sc = scenes.vertex_processor_test_scene()
    v = sc.vertices + rng.normal(0, 0.03, sc.vertices.shape)
    v[:, 3:] = np.clip(v[:, 3:], 0.0, 1.0)
    return scenes.Scene(v.astype(np.float32), sc.indices, sc.mvp, w, h)


class UvVertexShader(api.VertexShaderBase):
    """clip = M * (p, 1), pvar = uv over {p, normal, uv}: the Box demo's vertex shader."""

    AttribCount, AVarCount, PVarCount = 1, 0, 2
    Program = api.VS_MVP_POS_UV

    def __init__(self, mvp):
        self.mvp = np.asarray(mvp, np.float32)


class Drawing:
    """A rasterizer with its state, its targets and their clear values, and the draw call."""

    def __init__(self, case, sc, host=False):
        self.host = host
        self.r = api.Rasterizer(0)
        self.v = api.VertexProcessor(self.r)
        h, w = case["height"], case["width"]
        self.size = (h, w)
        self.r.setScissorRect(0, 0, w, h)
        self.v.setViewport(0, 0, w, h)
        self.vertices = sc.vertices if host else torch.from_numpy(sc.vertices).cuda()
        self.indices = sc.indices if host else torch.from_numpy(sc.indices).cuda()
        self.stride = sc.stride
        self.targets, self.values = [], []

    def target(self, dtype, value):
        if self.host:
            t = np.full(self.size, value, {torch.int32: np.int32, torch.float32: np.float32}[dtype])
        else:
            t = torch.full(self.size, value, dtype=dtype, device="cuda")
        self.targets.append(t)
        self.values.append(value)
        return t

    def clear(self):
        for t, x in zip(self.targets, self.values):
            t.fill(x) if self.host else t.fill_(x)

    def __del__(self):  # a texture goes before the context that made it
        texture = getattr(self, "texture", None)
        if texture is not None:
            texture.close()
        self.r.close()

    def bind(self, vshader, pshader):
        self.v.setVertexShader(vshader)
        self.v.setVertexAttribPointer(0, self.stride, self.vertices)
        self.r.setPixelShader(pshader)


def _pixel_program(d, name):
    if name == "depth":
        return api.DepthCheckerShader(d.target(torch.int32, 0), d.target(torch.float32, 1.0))
    if name == "visibility":
        return api.VisibilityShader(d.target(torch.int32, 0), d.target(torch.float32, 1.0))
    if name == "hash":
        return api.HashShader(d.target(torch.int32, -2128831035), d.target(torch.int32, 0))
    if name == "coverage":
        return api.CoverageShader(d.target(torch.int32, 0))
    return api.RGBShader(d.target(torch.int32, 0))


def _prepare_frame(case, seed):
    sc = _scene(case, seed)
    d = Drawing(case, sc, case["host"])
    ps = _pixel_program(d, case["program"])
    d.r.setRasterMode(case["mode"])
    d.v.setCullMode(case["cull"])
    vs = {"overdraw": api.PosRGBVertexShader, "triangle": api.PosRGBVertexShader,
          "clip": lambda: api.RawVertexShader(3, 2)}.get(
              case["scene"], lambda: api.MvpVertexShader(sc.mvp))()
    if case["tuned"]:  # what the autotuner leaves set for the full-HD soup
        d.r.setTuning(bin_size=16, waves_per_bin=4, expand_chunk=512, vertex_pass=-1)
    d.bind(vs, ps)
    d.v.drawElements(api.DrawMode.Triangle, d.indices)  # sizes the arenas for async draws
    draw_call = d.v.drawElements if case["sync"] else d.v.drawElementsAsync

    def step():
        d.clear()
        draw_call(api.DrawMode.Triangle, d.indices)
        return d.targets

    return d, step


def _prepare_texture(case, seed):
    if case["scene"] == "floor":
        rng = np.random.default_rng(seed)
        sc = scenes.floor_scene(case["width"], case["height"], extent=rng.uniform(18, 24),
                                repeat=rng.uniform(12, 20))
    else:
        sc = _sphere(case, seed)
    d = Drawing(case, sc)
    tex = api.Texture(d.r, scenes.procedural_texture("noise", case["texels"], case["texels"], seed),
                      max_anisotropy=case["aniso"])
    d.r.setRasterMode(case["mode"])
    d.v.setCullMode(CW)
    d.texture = tex
    d.bind(UvVertexShader(sc.mvp), api.TextureShader(d.target(torch.int32, 0), tex))
    d.v.drawElements(api.DrawMode.Triangle, d.indices)

    def step():
        d.clear()
        d.v.drawElementsAsync(api.DrawMode.Triangle, d.indices)
        return d.targets

    return d, step


def _prepare_lines(case, seed):
    line = case["draw"] == "line"
    mode = api.DrawMode.Line if line else api.DrawMode.Point
    if case["scene"] == "wire":  # a mesh's edges or vertices through the vertex processor
        sc = _sphere(dict(case, tris=max(50, case["count"] // 3)), seed)
        d = Drawing(case, sc)
        idx = scenes.edge_indices(sc.indices) if line else sc.indices
        d.indices = torch.from_numpy(idx).cuda()
        d.bind(api.MvpVertexShader(sc.mvp), _pixel_program(d, "depth"))

        def step():
            d.clear()
            d.v.drawElements(mode, d.indices)
            return d.targets
    else:  # window-space lists through the rasterizer's own entry points
        v = scenes.window_lines(case["count"], seed, case["width"], case["height"])
        d = Drawing(case, scenes.Scene(np.zeros((1, 8), np.float32), np.zeros(3, np.int32),
                                       np.eye(4), case["width"], case["height"]))
        verts = torch.from_numpy(v.view(np.float32).reshape(-1, 36)).cuda()
        idx = torch.arange(verts.shape[0], dtype=torch.int32, device="cuda")
        d.r.setPixelShader(_pixel_program(d, "depth"))
        call = d.r.drawLineList if line else d.r.drawPointList

        def step():
            d.clear()
            call(verts, idx)
            return d.targets
    return d, step


def _batch_scenes(case, seed):
    """Sizes and modes are the case's own (independent of the seed), colours the seed's."""
    rng = np.random.default_rng(case["scenes"] * 7919 + case["hi"])
    out = []
    for i in range(case["scenes"]):
        t = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        w, h = scenes.BATCH_SIZES[int(rng.integers(len(scenes.BATCH_SIZES)))]
        mode = int(rng.integers(2))
        n = _rings(t)
        if seed is None:
            out.append((n, w, h))
        else:
            sc = scenes.sphere_scene(n, 2 * n, seed=seed * 1000 + i, width=w, height=h)
            sc.info["raster_mode"] = mode
            out.append(sc)
    return out


def _prepare_batch(case, seed):
    work = _batch_scenes(case, seed)
    px = np.concatenate([[0], np.cumsum([s.width * s.height for s in work])])
    color = torch.zeros(int(px[-1]), dtype=torch.int32, device="cuda")
    depth = torch.ones(int(px[-1]), dtype=torch.float32, device="cuda")
    r = api.Rasterizer(0)
    v = api.VertexProcessor(r)
    v.setVertexShader(api.MvpVertexShader(work[0].mvp))
    tg = [(color[a:b].view(s.height, s.width), depth[a:b].view(s.height, s.width))
          for s, a, b in zip(work, px, px[1:])]
    r.setPixelShader(api.DepthCheckerShader(*tg[0]))
    batch = api.Batch(r, [
        dict(indices=torch.from_numpy(s.indices).cuda(),
             vertices=torch.from_numpy(s.vertices).cuda(), stride=s.stride, mvp=s.mvp,
             viewport=(0, 0, s.width, s.height), scissor=(0, 0, s.width, s.height), cull_mode=CW,
             raster_mode=s.info["raster_mode"], targets=t, size=(s.height, s.width))
        for s, t in zip(work, tg)])
    batch.draw()

    def step():
        color.zero_()
        depth.fill_(1.0)
        batch.draw(async_=True)
        return [color, depth]

    return (r, v, batch), step


@functools.lru_cache(maxsize=None)
def _icosphere(subdiv):
    return scenes.icosphere(subdiv)


def _target(views, size, channels, seed):
    """A blocky random photograph per view, [views, size, size, channels]."""
    rng = np.random.default_rng(seed + 17)
    low = torch.from_numpy(rng.random((views, channels, 16, 16), dtype=np.float32)).cuda()
    up = torch.nn.functional.interpolate(low, size=(size, size), mode="nearest")
    return up.permute(0, 2, 3, 1).contiguous()


def _diff_inputs(case, seed):
    """(triangles, clip [V, N, 4] fp32, attributes [N, C] fp32, target) of a mesh in view."""
    pos, tris = _icosphere(case["subdiv"])
    rng = np.random.default_rng(seed)
    pos = pos * rng.uniform(0.8, 1.1) * (1.0 + 0.02 * rng.standard_normal((pos.shape[0], 1))
                                         * 4.0 ** (3 - max(case["subdiv"], 3)))
    hom = np.concatenate([pos, np.ones((pos.shape[0], 1))], 1)
    mvps = scenes.orbit_cameras(case["views"], case["size"], case["size"], seed=seed)
    clip = np.matmul(hom, mvps.transpose(0, 2, 1)).astype(np.float32)
    attr = rng.random((pos.shape[0], case["channels"])).astype(np.float32)
    return (tris, torch.from_numpy(clip).cuda(), torch.from_numpy(attr).cuda(),
            _target(case["views"], case["size"], case["channels"], seed))


def _prepare_diff(case, seed):
    tris, clip, attr, target = _diff_inputs(case, seed)
    r = diff.DiffRenderer(tris, attr.shape[0], case["views"], case["size"], case["size"],
                          channels=case["channels"])
    r.forward(clip, attr, sync=True)  # sizes the arenas
    if case["api"] == "autograd":
        clip.requires_grad_(True)
        attr.requires_grad_(True)

        def step():
            image = diff.render(r, clip, attr)
            loss = 0.5 * ((image - target) ** 2).sum()
            gclip, gattr = torch.autograd.grad(loss, [clip, attr])
            return {"image": image.detach(), "gclip": gclip, "gattr": gattr}
    else:

        def step():
            image = r.forward(clip, attr)
            gclip, gattr = r.backward_l2(target)
            return {"image": image, "gclip": gclip, "gattr": gattr}

    return r, step


def _cells(case):
    rng = np.random.default_rng(case["scenes"] * 7919 + case["hi"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [int(round(math.exp(rng.uniform(lo, hi)))) for _ in range(case["scenes"])]


def _prepare_terrain(case, seed):
    size, views = case["size"], case["views"]
    work, clips, cols = [], [], []
    for k, cells in enumerate(_cells(case)):
        pos, tris, col = scenes.heightfield(cells, seed=seed * 1000 + k)
        mvps = scenes.terrain_cameras(views, size, size, seed=seed * 1000 + k)
        hom = np.concatenate([pos, np.ones((pos.shape[0], 1))], 1)
        clips.append(torch.from_numpy(np.matmul(hom, mvps.transpose(0, 2, 1)).astype(np.float32)))
        cols.append(torch.from_numpy(col.astype(np.float32)))
        work.append((tris, pos.shape[0], views))
    r = diff.SceneDiffRenderer(work, size, size)
    clip = diff.SceneDiffRenderer.clip_rows(clips).cuda()
    attr = torch.cat(cols).cuda()
    target = _target(r.V, size, 3, seed)
    r.forward(clip, attr, sync=True)

    def step():
        image = r.forward(clip, attr)
        gclip, gattr = r.backward(image - target)
        return {"image": image, "gclip": gclip, "gattr": gattr}

    return r, step


def prepare(case, seed):
    make = {"frame": _prepare_frame, "texture": _prepare_texture, "lines": _prepare_lines,
            "batch": _prepare_batch, "diff": _prepare_diff, "terrain": _prepare_terrain}
    return make[case["kind"]](case, seed)


def run(state):
    _, step = state
    return step()


# ---- what a pass cannot do without -------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("frame", "texture", "lines"):
        px = case["width"] * case["height"]
        if kind == "lines":
            n = case["count"]
            if case["scene"] == "wire":  # two indices per edge, shared 32-byte vertices
                data, ops = 8 * n + 32 * n // 6, 60 * n
            else:  # two 144-byte window vertices per line
                data, ops = 2 * (4 + 144) * n, 60 * n
            return {"bytes": data + 16 * px, "flops": ops}
        t = case["tris"]
        verts = {"soup": 2.1 * t, "sphere": 0.5 * t, "floor": 4}.get(case["scene"], 3 * t)
        stride = {"overdraw": 24, "triangle": 24, "clip": 36}.get(case["scene"], 32)
        planes = {"depth": 16, "visibility": 16, "hash": 16}.get(case.get("program"), 8)
        # indices and vertices read, targets cleared (or read) and written; a transform per
        # vertex, a setup per triangle, an interpolation per pixel
        return {"bytes": 12 * t + stride * verts + planes * px,
                "flops": 32 * verts + 100 * t + 40 * px}
    if kind == "batch":
        b = f = 0
        for n, w, h in _batch_scenes(case, None):
            t = 4 * n * (n - 1)
            b += 12 * t + 16 * t + 16 * w * h
            f += 116 * t + 40 * w * h
        return {"bytes": b, "flops": f}
    if kind == "diff":
        n, t, v, c = 10 * 4 ** case["subdiv"] + 2, 20 * 4 ** case["subdiv"], case["views"], case["channels"]
        px = v * case["size"] ** 2
    else:
        cells, v, c = _cells(case), case["scenes"] * case["views"], 3
        n, t = sum((k + 1) ** 2 for k in cells) * case["views"] / v, sum(2 * k * k for k in cells) * case["views"] / v
        px = v * case["size"] ** 2
    # clip rows read and their gradients written, per view; triangles once per view; image
    # written, target read; attributes and their gradients
    return {"bytes": v * n * 32 + v * t * 12 + px * 8 * c + n * c * 8,
            "flops": v * t * 100 + px * (120 + 60 * c)}


# ---- the differentiable renderer in 64 bits ----------------------------------------------


def _visible(win, z, tris, size):
    """(triangle [size, size] (-1: none), depth): the nearest front-facing triangle at each
    pixel, which is a matter of fp32 rules: the Span coverage of window positions win [N, 2],
    and window depths z [N] stepped along each span."""
    dev = win.device
    a, b, c = (win[tris[:, k]] for k in range(3))
    facing = (a[:, 0] - b[:, 0]) * (c[:, 1] - b[:, 1]) - (c[:, 0] - b[:, 0]) * (a[:, 1] - b[:, 1])
    keep = torch.nonzero(facing > 0)[:, 0]
    v = torch.stack([c[keep], b[keep], a[keep]], 1)  # the cull swaps the first and the last
    zt = z[tris[keep]].flip(1)
    # the depth plane, from the edge equations
    eq = []
    for i, j in ((1, 2), (2, 0), (0, 1)):
        ea, eb = v[:, i, 1] - v[:, j, 1], v[:, j, 0] - v[:, i, 0]
        eq.append((ea, eb, -(ea * (v[:, i, 0] + v[:, j, 0]) + eb * (v[:, i, 1] + v[:, j, 1])) / 2))
    f = 1.0 / (eq[0][2] + eq[1][2] + eq[2][2])
    plane = [f * (zt[:, 0] * eq[0][n] + zt[:, 1] * eq[1][n] + zt[:, 2] * eq[2][n])
             for n in range(3)]
    t, m, o = v.unbind(1)
    for x, y in ((0, 1), (1, 2), (0, 1)):  # by y, ties as they are
        p = [t, m, o]
        sw = (p[x][:, 1] > p[y][:, 1])[:, None]
        p[x], p[y] = torch.where(sw, p[y], p[x]), torch.where(sw, p[x], p[y])
        t, m, o = p
    flat_top, flat_bot = m[:, 1] == t[:, 1], m[:, 1] == o[:, 1]
    split = torch.stack([t[:, 0] + ((o[:, 0] - t[:, 0]) / (o[:, 1] - t[:, 1])) *
                         (m[:, 1] - t[:, 1]), m[:, 1]], 1)
    other = torch.where(flat_top[:, None], t, torch.where(flat_bot[:, None], o, split))
    sw = (m[:, 0] > other[:, 0])[:, None]
    l, r = torch.where(sw, other, m), torch.where(sw, m, other)
    trunc = lambda f: f.nan_to_num(0.0).clamp(-1e6, 1e6).trunc().long()  # noqa: E731
    parts = [  # apex, slopes, first and last row
        (t, (l[:, 0] - t[:, 0]) / (l[:, 1] - t[:, 1]), (r[:, 0] - t[:, 0]) / (r[:, 1] - t[:, 1]),
         trunc(t[:, 1] + 0.5), trunc(l[:, 1] + 0.5) - 1, ~flat_top),
        (o, (o[:, 0] - l[:, 0]) / (o[:, 1] - l[:, 1]), (o[:, 0] - r[:, 0]) / (o[:, 1] - r[:, 1]),
         trunc(l[:, 1] - 0.5) + 1, trunc(o[:, 1] - 0.5), ~(flat_bot & ~flat_top))]
    hits = []
    for apex, s1, s2, y0, y1, on in parts:
        rows = int((y1 - y0).max().clamp(min=-1)) + 1
        y = y0[:, None] + torch.arange(rows, device=dev)
        ok = on[:, None] & (y <= y1[:, None]) & (y >= 0) & (y < size)
        dy = (y.float() - apex[:, 1:]) + 0.5
        xl = trunc(apex[:, :1] + s1[:, None] * dy + 0.5).clamp(min=0)
        xr = trunc(apex[:, :1] + s2[:, None] * dy + 0.5).clamp(max=size)
        k, row = torch.nonzero(ok & (xl < xr), as_tuple=True)
        n = (xr - xl)[k, row]
        rep = torch.repeat_interleave(torch.arange(k.numel(), device=dev), n)
        at = torch.arange(rep.numel(), device=dev) - (torch.cumsum(n, 0) - n)[rep]
        x0, ys, kk = xl[k, row][rep], y[k, row][rep], k[rep]
        pa = plane[0][kk]
        zp = pa * (x0.float() + 0.5) + plane[1][kk] * (ys.float() + 0.5) + plane[2][kk]
        for s in range(int(at.max()) if at.numel() else 0):
            zp = torch.where(at > s, zp + pa, zp)
        hits.append((kk, ys * size + x0 + at, zp))
    k, pix, zp = (torch.cat(h) for h in zip(*hits))
    tri = keep[k]
    depth = torch.ones(size * size, dtype=torch.float32, device=dev)
    depth.scatter_reduce_(0, pix, zp, "amin")
    ids = torch.full((size * size,), 1 << 40, device=dev)
    won = (zp == depth[pix]) & (zp < 1.0)
    ids.scatter_reduce_(0, pix[won], tri[won], "amin")
    ids[ids == 1 << 40] = -1
    return ids.view(size, size), depth.view(size, size)


def _adjacent(tris):
    """[T, 3]: the triangle across the edge opposite each vertex of a closed mesh."""
    t = np.asarray(tris, np.int64)
    e = np.sort(np.stack([t[:, [1, 2]], t[:, [2, 0]], t[:, [0, 1]]], 1).reshape(-1, 2), 1)
    order = np.lexsort((e[:, 1], e[:, 0]))
    adj = np.empty(3 * len(t), np.int64)
    adj[order[0::2]], adj[order[1::2]] = order[1::2] // 3, order[0::2] // 3
    return adj.reshape(-1, 3)


def _edge(j, k, p):
    return (k[:, 0] - j[:, 0]) * (p[:, 1] - j[:, 1]) - (k[:, 1] - j[:, 1]) * (p[:, 0] - j[:, 0])


def _crossings(ids, depth, win, tris, adj, dx, dy):
    """The silhouette crossings between every pixel and its (dx, dy) neighbour: (front pixel,
    other pixel, low half?, triangle, edge vertices j, k, orientation)."""
    size = ids.shape[0]
    grid = torch.arange(size * size, device=ids.device).view(size, size)
    p, q = grid[:size - dy, :size - dx].reshape(-1), grid[dy:, dx:].reshape(-1)
    f = ids.view(-1)
    a, b = f[p], f[q]
    shared = (tris[a.clamp(min=0)][:, :, None] == tris[b.clamp(min=0)][:, None, :]).any(2).any(1)
    todo = (a != b) & ~((a >= 0) & (b >= 0) & shared)
    p, q, a, b = p[todo], q[todo], a[todo], b[todo]
    dp, dq = depth.view(-1)[p], depth.view(-1)[q]
    pf = (a >= 0) & ((b < 0) | (dp <= dq))
    front, back, cur = torch.where(pf, p, q), torch.where(pf, q, p), torch.where(pf, a, b)
    centre = lambda i: torch.stack([i % size, i // size], 1).float() + 0.5  # noqa: E731
    done, came = [], torch.full_like(cur, -1)
    for _ in range(8):
        if not cur.numel():
            break
        F, Q = centre(front), centre(back)
        v = win[tris[cur]]
        s = torch.sign(_edge(v[:, 0], v[:, 1], v[:, 2]))
        best, out = torch.full_like(s, 2.0), torch.full_like(cur, -1)
        for e in range(3):
            j, k = v[:, (e + 1) % 3], v[:, (e + 2) % 3]
            ef, eq = s * _edge(j, k, F), s * _edge(j, k, Q)
            t = ef / (ef - eq)
            hit = (came != e) & (eq < 0) & (ef > eq) & (t < best)
            best, out = torch.where(hit, t, best), torch.where(hit, e, out)
        nxt = adj[cur, out.clamp(min=0)]
        nv = win[tris[nxt]]
        inner = torch.sign(_edge(nv[:, 0], nv[:, 1], nv[:, 2])) == s
        end = (out >= 0) & ~inner
        j = tris[cur, (out + 1) % 3]
        k = tris[cur, (out + 2) % 3]
        done.append((front[end], back[end], best[end] < 0.5, cur[end], j[end], k[end], s[end]))
        go = (out >= 0) & inner
        came = (adj[nxt] == cur[:, None]).float().argmax(1)[go]
        front, back, cur = front[go], back[go], nxt[go]
    return [torch.cat(x) for x in zip(*done)] if done else None


def _shade(clip, attr, tri, ndc, tris):
    """Attributes at rays (ndc, 1) of triangles `tri`: perspective-correct, fp64."""
    h = clip[tris[tri]][..., [0, 1, 3]]
    r = torch.cat([ndc, torch.ones_like(ndc[:, :1])], 1)
    D = torch.stack([(r * torch.linalg.cross(h[:, (m + 1) % 3], h[:, (m + 2) % 3])).sum(1)
                     for m in range(3)], 1)
    return ((D / D.sum(1, keepdim=True))[..., None] * attr[tris[tri]]).sum(1)


def _view_image(clip, attr, tris, adj, size):
    """One view's image [size, size, C] in fp64, differentiable in clip and attr."""
    c = clip.detach().float()
    half = size / 2.0
    inv = 1.0 / c[:, 3]
    draw_win = torch.stack([half * (c[:, 0] * inv) + half, half * -(c[:, 1] * inv) + half], 1)
    ids, depth = _visible(draw_win, 0.5 * (c[:, 2] * inv) + 0.5, tris, size)
    walk_win = torch.stack([half * (c[:, 0] / c[:, 3]) + half,
                            -half * (c[:, 1] / c[:, 3]) + half], 1)
    to_ndc = lambda P: torch.stack([2 * P[:, 0] / size - 1, 1 - 2 * P[:, 1] / size], 1)  # noqa: E731
    centre = lambda i: torch.stack([i % size, i // size], 1).double() + 0.5  # noqa: E731
    flat = ids.view(-1)
    seen = torch.nonzero(flat >= 0)[:, 0]
    color = torch.zeros(size * size, attr.shape[1], dtype=torch.float64, device=clip.device)
    color = color.index_copy(0, seen, _shade(clip, attr, flat[seen], to_ndc(centre(seen)), tris))
    image = color
    win = torch.stack([half * (clip[:, 0] / clip[:, 3]) + half,
                       -half * (clip[:, 1] / clip[:, 3]) + half], 1)
    for dx, dy in ((1, 0), (0, 1)):
        got = _crossings(ids, depth, walk_win, tris, adj, dx, dy)
        if got is None or not got[0].numel():
            continue
        front, back, low, tri, j, k, s = got
        F, Q = centre(front), centre(back)
        ef, eq = s * _edge(win[j], win[k], F), s * _edge(win[j], win[k], Q)
        t = ef / (ef - eq)
        e = win[k] - win[j]
        axis = (e[:, 1] if dx else e[:, 0]) ** 2 / (e ** 2).sum(1)
        mix = (axis * (0.5 - t))[:, None] * (color[back] - color[front])
        image = image.index_add(0, front[low], mix[low])
        hi = ~low
        E = _shade(clip, attr, tri[hi], to_ndc(F[hi] + t[hi, None] * (Q - F)[hi]), tris)
        image = image.index_add(0, back[hi], (axis * (t - 0.5))[hi, None] * (E - color[back[hi]]))
    return image.view(size, size, -1)


def exact(case, seed):
    if case["kind"] == "terrain":
        return None  # clipped triangles and megapixel views: minutes in plain torch
    if case["kind"] != "diff":
        return None  # bits, not rounded values
    faces, clip32, attr32, target = _diff_inputs(case, seed)
    tris = torch.from_numpy(np.asarray(faces, np.int64)).to(clip32.device)
    adj = torch.from_numpy(_adjacent(faces)).to(clip32.device)
    attr = attr32.double().requires_grad_(True)
    images, gclip, gattr = [], [], torch.zeros_like(attr32, dtype=torch.float64)
    for v in range(case["views"]):
        clip = clip32[v].double().requires_grad_(True)
        image = _view_image(clip, attr, tris, adj, case["size"])
        loss = 0.5 * ((image - target[v].double()) ** 2).sum()
        gc, ga = torch.autograd.grad(loss, [clip, attr])
        images.append(image.detach())
        gclip.append(gc)
        gattr += ga
    return {"image": torch.stack(images), "gclip": torch.stack(gclip), "gattr": gattr}
