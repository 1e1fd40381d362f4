"""The work that programs built on this rasterizer have it do, as timed cases.

Every case is one pass through the public Python front end: plain draws
(`CudaRaster`), a whole demo frame, texPhong draws, batched views (`Batch`),
differentiable views (`DiffRasterizer`) and the vertex shader.  Inputs are
seeded and made on the GPU.  Distributions are those of
`cudaraster.scenes`: independent triangles with centres uniform over the
viewport, log-uniform screen areas, random winding (half are back-facing) and
random eye depths; for single differentiable views also a connected mesh, the
usual input of an optimisation loop.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cudaraster-linux_amd"))
import cudaraster  # noqa: E402
from cudaraster import scenes  # noqa: E402
from cudaraster.diff import DiffRasterizer  # noqa: E402

BLENDS = {"replace": cudaraster.BLEND_REPLACE, "src_over": cudaraster.BLEND_SRC_OVER,
          "additive": cudaraster.BLEND_ADDITIVE, "depth_only": cudaraster.BLEND_DEPTH_ONLY}
LIT = cudaraster.RENDER_DEPTH | cudaraster.RENDER_LERP
CLEAR = (0.2, 0.4, 0.8, 1.0)


def plain(name, tris, width, height, samples_log2, blend="replace", ids=True, mode="sync", big=0,
          area_min=0.5, area_max=256.0):
    return {"name": name, "kind": "draw", "tris": tris, "big": big, "width": width, "height": height,
            "samples_log2": samples_log2, "blend": blend, "ids": ids, "mode": mode, "area_min": area_min,
            "area_max": area_max}


def listed():
    return [
        # The demo's 12-triangle cube: a draw that is all fixed cost.
        {"name": "cube", "kind": "cube", "width": 1024, "height": 768, "samples_log2": 0},
        # A small viewport of odd size drawn asynchronously, as a server with
        # a frame in flight does; colour and depth only.
        plain("draw_30k_async", 30_000, 1283, 717, 0, ids=False, mode="async"),
        # The headline workload: 1M triangles, 2048x2048, 4x MSAA.
        plain("draw_1m_4x", 1_000_000, 2048, 2048, 2),
        # Sub-pixel triangles under 1024 near-full-screen translucent ones.
        plain("draw_skewed_8x", 4_000_000, 2048, 2048, 3, blend="src_over", big=1024, area_min=0.05, area_max=1.0),
        # A demo frame: vertex shader, opaque draw, translucent draw over it, resolve.
        {"name": "frame_1080p_4x", "kind": "frame", "opaque": 300_000, "translucent": 50_000, "width": 1920,
         "height": 1080, "samples_log2": 2},
        # Textured Phong with quad derivatives.
        {"name": "tex_phong_4x", "kind": "phong", "tris": 20_000, "width": 1024, "height": 768, "samples_log2": 2,
         "quads": True},
        # A few small views at once (thumbnails, observations of an agent).
        {"name": "batch_8_small", "kind": "batch", "views": 8, "tris_min": 2_000, "tris_max": 20_000,
         "size_max": 256},
        # Views of the batched workload: 256x256 to 2048x2048, 1x and 4x.
        {"name": "batch_20", "kind": "batch", "views": 20, "tris_min": 10_000, "tris_max": 500_000,
         "size_max": 2048},
        # Differentiable views, forward and backward: 512x512, 200k triangles, 8 channels.
        {"name": "diff_views_16", "kind": "diff_views", "views": 16, "tris": 200_000, "width": 512, "height": 512,
         "channels": 8},
        # One view of a connected mesh (texture coordinates + a scalar), as a fitting loop renders it.
        {"name": "diff_mesh", "kind": "diff_render", "tris": 40_000, "width": 400, "height": 300, "channels": 3},
        # Many channels over an id image that is already there; reproducible gradients.
        {"name": "diff_ids_reproducible", "kind": "diff_ids", "tris": 100_000, "width": 640, "height": 480,
         "channels": 12, "deterministic": True},
        # The vertex shader over the headline workload's vertices, into 32-byte records.
        {"name": "vertex_3m", "kind": "vertex", "vertices": 3_000_000, "stride": 32},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def size(lo=64, hi=2048):
        return log_int(lo, hi), log_int(lo, hi)

    kind = rng.choice(("draw", "draw", "draw", "frame", "phong", "batch", "batch", "diff_views", "diff_views",
                       "diff_render", "diff_ids", "vertex"))
    w, h = size()
    if kind == "draw":
        blend = rng.choice(("replace", "replace", "src_over", "additive", "depth_only"))
        return {"kind": kind, "tris": log_int(12, min(1_000_000, w * h // 2)), "big": rng.choice((0, 0, 0, 64)),
                "width": w, "height": h, "samples_log2": rng.randrange(4), "blend": blend,
                "ids": rng.random() < 0.5, "mode": rng.choice(("sync", "sync", "async")), "area_min": 0.5,
                "area_max": 256.0}
    if kind == "frame":
        return {"kind": kind, "opaque": log_int(1_000, min(500_000, w * h)),
                "translucent": log_int(100, min(50_000, w * h // 4)), "width": w, "height": h,
                "samples_log2": rng.randrange(4)}
    if kind == "phong":
        return {"kind": kind, "tris": log_int(100, min(20_000, w * h // 32)), "width": w, "height": h,
                "samples_log2": rng.randrange(3), "quads": rng.random() < 0.5}
    if kind == "batch":
        n = rng.choice((2, 5, 8, 16, 20))
        return {"kind": kind, "views": n, "tris_min": log_int(500, 10_000), "tris_max": log_int(20_000, 400_000),
                "size_max": rng.choice((256, 512, 1024, 2048))}
    if kind == "vertex":
        return {"kind": kind, "vertices": log_int(1_000, 3_000_000), "stride": rng.choice((16, 32, 64))}
    w, h = size(64, 640)
    case = {"kind": kind, "tris": log_int(500, min(200_000, w * h)), "width": w, "height": h,
            "channels": rng.choice((1, 2, 3, 4, 8, 12, 16))}
    if kind == "diff_views":
        case["views"] = rng.choice((2, 4, 8, 16))
        case["channels"] = rng.choice((1, 3, 4, 8))
    else:
        case["deterministic"] = rng.random() < 0.4
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

class Seeded:
    """Uniform and normal device tensors from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def rand(self, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda")

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * self.rand(*shape)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.gen, device="cuda")


def project(px, py, w, width, height):
    """Pixel positions (y up) at eye depth w -> clip positions [..., 4], the demo camera's depth range."""
    far, near = scenes.ZFAR, scenes.ZNEAR
    z = (far + near) / (far - near) * w - 2.0 * far * near / (far - near)
    return torch.stack([(px / width * 2.0 - 1.0) * w, (py / height * 2.0 - 1.0) * w, z, w], -1)


def soup(g, n, width, height, area_min=0.5, area_max=256.0, depth=(scenes.ZNEAR, scenes.ZFAR)):
    """Clip positions [3n, 4] of n independent triangles (scenes.random_tris' distribution)."""
    cx, cy = g.uniform(0, width, n, 1), g.uniform(0, height, n, 1)
    area = torch.exp(g.uniform(math.log(area_min), math.log(area_max), n))
    third = torch.arange(3, device="cuda") * (2.0 * math.pi / 3.0)
    ang = g.uniform(0, 2.0 * math.pi, n, 1) + third + g.uniform(-math.pi / 6.0, math.pi / 6.0, n, 3)
    rad = g.uniform(0.6, 1.0, n, 3)
    x, y = rad * torch.cos(ang), rad * torch.sin(ang)
    flip = (g.rand(n, 1) < 0.5)
    x, y = torch.where(flip, x.flip(1), x), torch.where(flip, y.flip(1), y)
    a0 = 0.5 * ((x[:, 1] - x[:, 0]) * (y[:, 2] - y[:, 0]) - (x[:, 2] - x[:, 0]) * (y[:, 1] - y[:, 0])).abs()
    s = torch.sqrt(area / a0.clamp(min=1e-9))[:, None]
    x, y = (x - x.mean(1, keepdim=True)) * s, (y - y.mean(1, keepdim=True)) * s
    w = (g.uniform(depth[0], depth[1], n, 1) * g.uniform(0.9, 1.1, n, 3)).clamp(depth[0], depth[1])
    return project(cx + x, cy + y, w, width, height).reshape(3 * n, 4)


def wide(g, n, width, height):
    """Clip positions [3n, 4] of n front-facing triangles spanning roughly the whole viewport."""
    base = torch.tensor([[-0.15, -0.15], [1.15, -0.10], [0.5, 1.2]], device="cuda")
    p = base + (g.rand(n, 3, 2) - 0.5) * 0.5
    w = (g.uniform(scenes.ZNEAR, scenes.ZFAR, n, 1) * g.uniform(0.9, 1.1, n, 3)).clamp(scenes.ZNEAR, scenes.ZFAR)
    return project(p[..., 0] * width, p[..., 1] * height, w, width, height).reshape(3 * n, 4)


def colours(g, vertices, alpha=(0.0, 1.0)):
    c = g.rand(vertices, 4)
    c[:, 3] = alpha[0] + (alpha[1] - alpha[0]) * c[:, 3]
    return c


def own_indices(n):
    return torch.arange(3 * n, dtype=torch.int32, device="cuda").reshape(n, 3)


def mixed(g, case):
    """The triangles of a plain draw: small ones, large ones dropped in between at random places."""
    n, nb, w, h = case["tris"], case["big"], case["width"], case["height"]
    clip = soup(g, n, w, h, case["area_min"], case["area_max"])
    if nb:
        clip = torch.cat([clip, wide(g, nb, w, h)]).reshape(n + nb, 3, 4)
        clip = clip[torch.randperm(n + nb, generator=g.gen, device="cuda")].reshape(-1, 4)
    alpha = (0.0, 1.0) if case["blend"] == "replace" else (0.2, 0.8)
    return torch.cat([clip, colours(g, clip.shape[0], alpha)], 1).contiguous(), own_indices(n + nb)


def mesh(g, tris, width, height):
    """A bumpy sheet of about `tris` connected triangles seen at a slant: clip positions [V, 4], indices [T, 3]."""
    nx = max(1, int(math.sqrt(tris / 2 * width / height)))
    ny = max(1, tris // (2 * nx))
    u = torch.linspace(-1.1, 1.1, nx + 1, device="cuda").expand(ny + 1, nx + 1)
    v = torch.linspace(-1.1, 1.1, ny + 1, device="cuda")[:, None].expand(ny + 1, nx + 1)
    f, p = g.uniform(2.0, 9.0, 4), g.uniform(0.0, 2.0 * math.pi, 4)
    bump = 0.15 * (torch.sin(f[0] * u + p[0]) * torch.sin(f[1] * v + p[1])) \
        + 0.05 * torch.sin(f[2] * 2 * u + p[2]) * torch.sin(f[3] * 2 * v + p[3])
    depth = 3.0 + 0.8 * v + bump
    px = (0.5 + 0.5 * u * 3.0 / depth) * width
    py = (0.5 + 0.45 * (v + 0.6 * bump) * 3.0 / depth) * height
    pos = project(px, py, depth, width, height).reshape(-1, 4).contiguous()
    i = torch.arange(nx, device="cuda")[None, :] + torch.arange(ny, device="cuda")[:, None] * (nx + 1)
    quad = torch.stack([i, i + 1, i + nx + 2, i, i + nx + 2, i + nx + 1], -1)
    return pos, quad.reshape(-1, 3).to(torch.int32).contiguous()


# ---------------------------------------------------------------------------
# Surfaces and draws
# ---------------------------------------------------------------------------

class DeviceWords:
    """A surface's texels for torch.as_tensor: the surface's own memory, no copy.  The tensor refers to this object
    and so keeps the surface, whose memory it shows, alive."""

    def __init__(self, surface):
        self.surface = surface
        ptr, _ = surface.device_ptr()
        self.__cuda_array_interface__ = {"shape": surface.shape, "typestr": "<i4", "data": (ptr, False),
                                         "version": 2}


class Target:
    """Colour, depth and, when wanted, triangle-id surfaces and their texels as tensors."""

    def __init__(self, width, height, samples_log2, ids=True):
        n = 1 << samples_log2
        formats = [cudaraster.FORMAT_RGBA8, cudaraster.FORMAT_DEPTH32] + [cudaraster.FORMAT_TRIANGLE_ID] * ids
        self.surfaces = [cudaraster.CudaSurface((width, height), f, n) for f in formats]
        self.texels = [torch.as_tensor(DeviceWords(s), device="cuda") for s in self.surfaces]

    def bind(self, cr):
        cr.setSurfaces(*self.surfaces[:2])
        cr.setTriangleIdSurface(self.surfaces[2] if len(self.surfaces) > 2 else None)


def prepare_draw(case, seed):
    g = Seeded(seed)
    target = Target(case["width"], case["height"], case["samples_log2"], case.get("ids", True))
    cr = cudaraster.CudaRaster().init()
    target.bind(cr)
    if case["kind"] == "cube":
        scene = scenes.cube(case["width"], case["height"], case["samples_log2"], seed=seed)
        verts, tris = cudaraster.device_buffers(scene)
    else:
        verts, tris = mixed(g, case)
    cr.setPixelPipe(cudaraster.pipe_desc(32, cudaraster.SHADER_GOURAUD, BLENDS[case.get("blend", "replace")],
                                         case["samples_log2"], LIT))
    cr.setVertexBuffer(verts)
    cr.setIndexBuffer(tris, 0, tris.shape[0])
    if case.get("mode") == "async":
        # A server draws its first frame synchronously, which sizes the queues.
        cr.deferredClear(CLEAR, 1.0)
        cr.drawTriangles(torch.cuda.current_stream())
    return {"kind": "draw", "mode": case.get("mode", "sync"), "cr": cr, "target": target}


def run_draw(s):
    cr, stream = s["cr"], torch.cuda.current_stream()
    if s["mode"] == "async":
        if cr.drawCheck() != cudaraster.CR_OK:            # the frame in flight, before the next one is queued
            raise RuntimeError("the frame before this one did not fit its queues")
        cr.deferredClear(CLEAR, 1.0)
        cr.drawTrianglesAsync(stream)
    else:
        cr.deferredClear(CLEAR, 1.0)
        cr.drawTriangles(stream)
    return s["target"].texels


def prepare_frame(case, seed):
    g = Seeded(seed)
    w, h, sl = case["width"], case["height"], case["samples_log2"]
    target = Target(w, h, sl)
    cr = cudaraster.CudaRaster().init()
    target.bind(cr)
    # Model positions whose clip positions under the camera below are the
    # usual triangles': undo the projection in 64 bits.
    camera = scenes.demo_camera(w, h)
    back = torch.from_numpy(np.linalg.inv(camera)).cuda()
    clip = soup(g, case["opaque"], w, h, depth=(1.0, 50.0)).double() @ back.T
    model = (clip[:, :3] / clip[:, 3:]).float().contiguous()
    opaque = torch.cat([torch.zeros_like(clip, dtype=torch.float32), colours(g, clip.shape[0])], 1).contiguous()
    clip2 = soup(g, case["translucent"], w, h, 4.0, 1024.0)
    translucent = torch.cat([clip2, colours(g, clip2.shape[0], (0.2, 0.8))], 1).contiguous()
    return {"kind": "frame", "cr": cr, "target": target, "camera": camera, "model": model, "opaque": opaque,
            "opaque_tris": own_indices(case["opaque"]), "translucent": translucent,
            "translucent_tris": own_indices(case["translucent"]),
            "opaque_pipe": cudaraster.pipe_desc(32, samples_log2=sl),
            "translucent_pipe": cudaraster.pipe_desc(32, blend_shader=cudaraster.BLEND_SRC_OVER, samples_log2=sl),
            "image": torch.empty((h, w), dtype=torch.int32, device="cuda")}


def run_frame(s):
    cr, stream = s["cr"], torch.cuda.current_stream()
    cr.vertexShaderPassthrough(s["model"], s["camera"], s["opaque"], out_stride=32, stream=stream)
    cr.setPixelPipe(s["opaque_pipe"])
    cr.setVertexBuffer(s["opaque"])
    cr.setIndexBuffer(s["opaque_tris"], 0, s["opaque_tris"].shape[0])
    cr.deferredClear(CLEAR, 1.0)
    cr.drawTriangles(stream)
    cr.setPixelPipe(s["translucent_pipe"])
    cr.setVertexBuffer(s["translucent"])
    cr.setIndexBuffer(s["translucent_tris"], 0, s["translucent_tris"].shape[0])
    cr.drawTriangles(stream)
    s["target"].surfaces[0].resolve(s["image"], stream)
    return [s["image"]] + s["target"].texels


def prepare_phong(case, seed):
    g = Seeded(seed)
    n, w, h = case["tris"], case["width"], case["height"]
    target = Target(w, h, case["samples_log2"])
    clip = soup(g, n, w, h, 4.0, 3000.0)
    depth = clip[:, 3:4]
    normal = g.normal(3 * n, 3)
    normal[:, 2] = -normal[:, 2].abs() - 0.3
    dense = torch.exp(g.uniform(math.log(0.05), math.log(20.0), n, 1, 1))
    uv = (g.uniform(-2.0, 2.0, n, 1, 2) + g.rand(n, 3, 2) * dense).reshape(3 * n, 2)
    one, zero = torch.ones_like(depth), torch.zeros_like(depth)
    verts = torch.cat([clip, clip[:, :2], -depth, one, normal, zero, uv, zero, one], 1).contiguous()
    # Materials and atlas as the texPhong scenes have them (two textures, an
    # alpha-tested material, an untextured one, one that is always discarded).
    look = scenes.tex_phong(1, seed=seed)
    cr = cudaraster.CudaRaster().init()
    target.bind(cr)
    flags = LIT | (cudaraster.RENDER_QUADS if case["quads"] else 0)
    cr.setPixelPipe(cudaraster.pipe_desc(64, cudaraster.SHADER_TEX_PHONG, samples_log2=case["samples_log2"],
                                         render_mode_flags=flags))
    cr.setShaderConstants(torch.from_numpy(look.materials.view(np.uint8).copy()).cuda(),
                          g.ints(4, n).to(torch.int32), torch.from_numpy(look.atlas).cuda())
    cr.setVertexBuffer(verts)
    cr.setIndexBuffer(own_indices(n), 0, n)
    return {"kind": "draw", "mode": "sync", "cr": cr, "target": target}


def batch_views(case):
    """Resolution, triangles and sample count of each view: a fixed spread over the case's ranges."""
    rng = np.random.default_rng(case["views"])
    sizes = [r for r in (64, 100, 256, 512, 1024, 2048) if case["size_max"] // 8 <= r <= case["size_max"]]
    lo, hi = math.log(case["tris_min"]), math.log(case["tris_max"])
    views = []
    for _ in range(case["views"]):
        r = int(rng.choice(sizes))
        views.append((r, int(math.exp(rng.uniform(lo, hi))), int(rng.choice((0, 2)))))
    return views


def prepare_batch(case, seed):
    g = Seeded(seed)
    cr = cudaraster.CudaRaster().init()
    targets, views, keep = [], [], []
    for size, n, sl in batch_views(case):
        t = Target(size, size, sl)
        clip = soup(g, n, size, size)
        verts, tris = torch.cat([clip, colours(g, 3 * n)], 1).contiguous(), own_indices(n)
        v = cudaraster.View()
        v.color, v.depth, v.tri_id = (f.handle.value for f in t.surfaces)
        v.vertices, v.num_vertices = verts.data_ptr(), verts.shape[0]
        v.indices, v.num_tris = tris.data_ptr(), n
        v.deferred_clear = 1
        v.pipe = cudaraster.pipe_desc(32, samples_log2=sl)
        v.clear_color[:] = CLEAR
        v.clear_depth = 1.0
        targets.append(t)
        views.append(v)
        keep += [verts, tris]
    batch = cudaraster.Batch(cr, views, keep)
    return {"kind": "batch", "cr": cr, "batch": batch, "targets": targets}


def prepare_diff(case, seed):
    g = Seeded(seed)
    n, w, h, c, kind = case.get("views", 1), case["width"], case["height"], case["channels"], case["kind"]
    pos, tris = [], []
    for _ in range(n):
        if kind == "diff_views":
            p, t = soup(g, case["tris"], w, h, depth=(1.0, 50.0)).contiguous(), own_indices(case["tris"])
        else:
            p, t = mesh(g, case["tris"], w, h)
        pos.append(p.requires_grad_(True))
        tris.append(t)
    attr = [g.uniform(-1.0, 1.0, p.shape[0], c).requires_grad_(True) for p in pos]
    shape = (n, h, w, c) if kind == "diff_views" else (h, w, c)
    state = {"kind": kind, "pos": pos, "attr": attr, "tris": tris, "upstream": g.normal(*shape),
             "raster": DiffRasterizer(w, h, deterministic=case.get("deterministic", False))}
    if kind == "diff_ids":
        state["ids"] = visible_ids(pos[0].detach(), tris[0], w, h).to(torch.int32)
    return state


def run_diff(s):
    raster, pos, attr, tris = s["raster"], s["pos"], s["attr"], s["tris"]
    if s["kind"] == "diff_views":
        image, ids = raster.render_views(pos, attr, tris)
    elif s["kind"] == "diff_ids":
        ids = None
        image = raster.render(pos[0], attr[0], tris[0], tri_image=s["ids"])
    else:
        ids = None
        image = raster.render(pos[0], attr[0], tris[0])
    grads = torch.autograd.grad(image, pos + attr, s["upstream"])
    return {"image": image, "ids": ids, "grads": list(grads)}


def prepare_vertex(case, seed):
    g = Seeded(seed)
    n = case["vertices"]
    cr = cudaraster.CudaRaster().init()
    model, out = g.normal(n, 3) * 20.0, g.rand(n, case["stride"] // 4)
    return {"kind": "vertex", "cr": cr, "model": model, "out": out, "stride": case["stride"],
            "camera": scenes.demo_camera(1920, 1080)}


def prepare(case, seed):
    by = {"cube": prepare_draw, "draw": prepare_draw, "frame": prepare_frame, "phong": prepare_phong,
          "batch": prepare_batch, "vertex": prepare_vertex}
    return by.get(case["kind"], prepare_diff)(case, seed)


def run(state):
    kind = state["kind"]
    if kind == "draw":
        return run_draw(state)
    if kind == "frame":
        return run_frame(state)
    if kind == "batch":
        state["batch"].draw(torch.cuda.current_stream())
        return [t.texels for t in state["targets"]]
    if kind == "vertex":
        state["cr"].vertexShaderPassthrough(state["model"], state["camera"], state["out"],
                                            out_stride=state["stride"], stream=torch.cuda.current_stream())
        return state["out"]
    return run_diff(state)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def rounded(size):
    return (size + 7) & ~7


def draw_bytes(tris, vertex_bytes, width, height, samples_log2, surfaces=3, read=False):
    """Vertex and index buffers read once, every surface written (and, without a clear, read) once."""
    texels = rounded(width) * rounded(height) << samples_log2
    return tris * (3 * vertex_bytes + 12) + texels * 4 * surfaces * (2 if read else 1)


def work(case):
    kind, w, h, sl = case["kind"], case.get("width"), case.get("height"), case.get("samples_log2")
    if kind == "cube":
        return {"bytes": draw_bytes(12, 32, w, h, sl), "flops": 0}
    if kind == "draw":
        surfaces = 2 + bool(case["ids"])
        return {"bytes": draw_bytes(case["tris"] + case["big"], 32, w, h, sl, surfaces), "flops": 0}
    if kind == "frame":
        return {"bytes": draw_bytes(case["opaque"], 12 + 32, w, h, sl) + w * h * 4
                + draw_bytes(case["translucent"], 32, w, h, sl, read=True), "flops": 0}
    if kind == "phong":
        return {"bytes": draw_bytes(case["tris"], 64, w, h, sl), "flops": 0}
    if kind == "batch":
        return {"bytes": sum(draw_bytes(n, 32, r, r, s) for r, n, s in batch_views(case)), "flops": 0}
    if kind == "vertex":
        return {"bytes": case["vertices"] * 28, "flops": case["vertices"] * 32}
    n, c = case.get("views", 1), case["channels"]
    verts = case["tris"] * 3 if kind == "diff_views" else case["tris"] // 2
    # Positions and attributes read and their gradients written; the image written, its gradient read.
    return {"bytes": n * (2 * verts * (16 + 4 * c) + 12 * case["tris"] + w * h * (8 * c + 4)),
            "flops": n * w * h * (60 + 18 * c)}


# ---------------------------------------------------------------------------
# The same values in 64 bits
# ---------------------------------------------------------------------------

def visible_ids(pos, tris, width, height):
    """Triangle id of every pixel [H, W] (-1: none), for triangles inside the depth range and the guard band:
    vertices snapped to 1/16 pixel, top-left rule at pixel centres, integer depth planes, first triangle of equal
    depth (the rules of cudaraster/cuda/TriangleSetup.inl:19-215 and Util.inl:65-91)."""
    f32, i64 = torch.float32, torch.int64
    v = pos[tris.long()]                                             # [T, 3, 4]
    rcp = (1.0 / v[..., 3].double()).to(f32)
    px = torch.round(v[..., 0] * rcp * float(width * 8)).to(i64) + width * 8
    py = torch.round(v[..., 1] * rcp * float(height * 8)).to(i64) + height * 8
    d1x, d1y, d2x, d2y = px[:, 1] - px[:, 0], py[:, 1] - py[:, 0], px[:, 2] - px[:, 0], py[:, 2] - py[:, 0]
    area = d1x * d2y - d1y * d2x
    # Depth plane.
    low, high = 2200 << 3, 0xFFFFFFFF - (2200 << 3)
    half, mid = float(np.float32(high - low)) * 0.5, float(np.float32(np.float32(high + low) * np.float32(0.5)))
    z = ((v[..., 2] * half).double() * rcp.double() + mid).to(f32)
    shift = ((z.amax(1).view(torch.int32).to(i64) >> 23) - 149).clamp(0, 8)
    t = z.double().clamp(0, 2.0 ** 32 - 1).to(i64) >> shift[:, None]
    t0, t1, t2 = t[:, 0], t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    bits = (1.0 / area.clamp(min=1).to(f32).double()).to(f32).view(torch.int32).to(i64)
    mantissa, rshift = (bits & 0x7FFFFF) | 0x800000, 150 - (bits >> 23)
    xc, yc = (t1 * d2y - t2 * d1y) * mantissa, (t2 * d1x - t1 * d2x) * mantissa
    zx, zy = xc >> (rshift - shift - 4), yc >> (rshift - shift - 4)
    x0, y0 = px[:, 0] - 8, py[:, 0] - 8
    zero = torch.zeros_like(d1x)
    cx = (2 * x0 + torch.minimum(torch.minimum(d1x, d2x), zero) + torch.maximum(torch.maximum(d1x, d2x), zero)) >> 5
    cy = (2 * y0 + torch.minimum(torch.minimum(d1y, d2y), zero) + torch.maximum(torch.maximum(d1y, d2y), zero)) >> 5
    cross = (xc >> 13) * (x0 - (cx << 4)) + (yc >> 13) * (y0 - (cy << 4))
    zb = (t0 << shift) - (cross >> (rshift - shift - 13)) - zx * cx - zy * cy
    # Every (triangle, pixel of its box) pair.
    bx0, bx1 = (px.amin(1) >> 4).clamp(min=0), (px.amax(1) >> 4).clamp(max=width - 1)
    by0, by1 = (py.amin(1) >> 4).clamp(min=0), (py.amax(1) >> 4).clamp(max=height - 1)
    bw, bh = (bx1 - bx0 + 1).clamp(min=0), (by1 - by0 + 1).clamp(min=0)
    count = torch.where(area > 0, bw * bh, zero)
    tri = torch.repeat_interleave(torch.arange(tris.shape[0], device=pos.device), count)
    rank = torch.arange(tri.shape[0], device=pos.device) - (torch.cumsum(count, 0) - count)[tri]
    x, y = bx0[tri] + rank % bw[tri], by0[tri] + rank // bw[tri]
    inside = torch.ones_like(tri, dtype=torch.bool)
    for k in range(3):
        dx, dy = px[:, (k + 1) % 3] - px[:, k], py[:, (k + 1) % 3] - py[:, k]
        open_edge = ((dy > 0) | ((dy == 0) & (dx <= 0))).to(i64)
        inside &= (px[tri, k] - 16 * x - 8) * dy[tri] - (py[tri, k] - 16 * y - 8) * dx[tri] - open_edge[tri] >= 0
    tri, x, y = tri[inside], x[inside], y[inside]
    depth = (zx[tri] * x + zy[tri] * y + zb[tri]) & 0xFFFFFFFF
    near = depth < high
    key = (depth * (1 << 24) + tri)[near]
    best = torch.full((height * width,), 1 << 60, dtype=i64, device=pos.device)
    best.scatter_reduce_(0, (y * width + x)[near], key, "amin")
    return torch.where(best < 1 << 60, best & 0xFFFFFF, torch.full_like(best, -1)).reshape(height, width)


def interpolated(pos, attr, tris, ids):
    """Perspective-correct attributes at pixel centres in 64 bits: image [H, W, C], 0 where no triangle is seen."""
    height, width = ids.shape
    y, x = torch.nonzero(ids >= 0, as_tuple=True)
    corner = tris[ids[y, x].long()].long()
    qx, qy = (2.0 * x + 1.0).double() / width - 1.0, (2.0 * y + 1.0).double() / height - 1.0
    v = pos[corner]                                                  # [P, 3, 4]
    xs, ys = v[..., 0] - qx[:, None] * v[..., 3], v[..., 1] - qy[:, None] * v[..., 3]
    c = xs.roll(-1, 1) * ys.roll(-2, 1) - ys.roll(-1, 1) * xs.roll(-2, 1)
    total = c.sum(1, keepdim=True)
    seen = total != 0
    b = torch.where(seen, c / torch.where(seen, total, torch.ones_like(total)), torch.zeros_like(c))
    image = torch.zeros((height, width, attr.shape[1]), dtype=torch.float64, device=pos.device)
    return image.index_put((y, x), (b[..., None] * attr[corner]).sum(1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "vertex":
        s = prepare_vertex(case, seed)
        out = s["out"].double()
        camera = torch.from_numpy(np.asarray(s["camera"], dtype=np.float32)).cuda().double()
        model = s["model"].double()
        out[:, :4] = torch.cat([model, torch.ones_like(model[:, :1])], 1) @ camera.T
        return out
    if not kind.startswith("diff"):
        return None                                                  # pixels: whole numbers
    s = prepare_diff(case, seed)
    n = len(s["pos"])
    pos = [p.detach().double().requires_grad_(True) for p in s["pos"]]
    attr = [a.detach().double().requires_grad_(True) for a in s["attr"]]
    upstream = s["upstream"].double().reshape(n, *s["upstream"].shape[-3:])
    images, gp, ga = [], [], []
    for k in range(n):
        ids = visible_ids(s["pos"][k].detach(), s["tris"][k], case["width"], case["height"])
        image = interpolated(pos[k], attr[k], s["tris"][k], ids)
        a, b = torch.autograd.grad(image, (pos[k], attr[k]), upstream[k])
        images.append(image.detach())
        gp.append(a)
        ga.append(b)
    image = torch.stack(images) if kind == "diff_views" else images[0]
    return {"image": image, "ids": None, "grads": gp + ga}
