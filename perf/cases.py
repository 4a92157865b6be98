"""The measured workloads: what programs have this renderer do, over the range
that they use.

Families:
  frame   one DrawModel::draw frame: clear, an optional shadow pass, the main
          pass, into a resident target
  viewer  such a frame, then the window's image on the host (hana_target_present)
  models  a cleared target, then one hana_draw per model, each with a mesh, a
          shader and uniforms of its own
  batch   many independent frames in one captured launch sequence
  micro   a frame of stacked grids whose triangles are a few pixels or less
  serve   a burst of requests to the render server, images on the host

A case's numbers fix the work (triangles, pixels, options); the seed draws
shapes, placement, cameras, lights and textures.  Colour is compared as bytes
and depth as the bits of its fp32 words: this renderer's depth is bit-exact by
contract, so both are whole numbers, which stay equal.  There is no 64-bit
value beside them: whether a pixel is covered at all is decided by the fp32
rounding that the contract fixes.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "hana-softwarerenderer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from hana_amd import gpu  # noqa: E402
from hana_amd import scenegen as sg  # noqa: E402

SHADERS = {"ground": sg.GROUND, "toon": sg.TOON, "texture": sg.TEXTURE, "texture_light": sg.TEXTURE_LIGHT,
           "blinn": sg.BLINN, "normalmap": sg.NORMALMAP}
# shaders whose material has a diffuse map; the normal map is NormalMap's alone
DIFFUSE = ("texture", "texture_light", "blinn", "normalmap")
MODEL_SHADERS = ("normalmap", "blinn", "texture_light", "texture", "toon", "ground")


def _frame(name, tris, width, height, shader, shadow=0, fp32=False, objects=1, dist=2.0, tex=512, family="frame"):
    """shadow: 0 none, -1 a frame-sized map (the renderer's default), else its edge."""
    return {"name": name, "family": family, "tris": tris, "objects": objects, "width": width, "height": height,
            "shader": shader, "shadow": shadow, "fp32": fp32, "dist": dist, "tex": tex}


def listed():
    return [
        # a thumbnail of a simple object: the smallest call, launches and latency
        _frame("thumbnail", 192, 128, 128, "toon"),
        # the plain small frame of the benchmark: a 4k-triangle sphere
        _frame("sphere", 3968, 800, 600, "normalmap", tex=1024),
        # the interactive application: a model of about 5,000 triangles in its
        # 1000x600 window, with its frame-sized shadow map, blitted each frame
        _frame("viewer", 5022, 1000, 600, "normalmap", shadow=-1, tex=1024, family="viewer"),
        # a room of models, one draw each, every shader, an odd-sized target
        {"name": "models", "family": "models", "tris": 60000, "objects": 12, "width": 1279, "height": 717, "tex": 256},
        # a mid-sized frame with the fp32 shadow-map option
        _frame("shaded", 60000, 1366, 768, "blinn", shadow=1024, fp32=True, objects=4, tex=1024),
        # the benchmark's single large frame
        _frame("large", 1310720, 1920, 1080, "normalmap", shadow=2048, tex=2048),
        # few large triangles on a large target: fill rate
        _frame("lowpoly", 300, 3840, 2160, "texture_light", objects=3, dist=1.6, tex=1024),
        # the camera dollied into the surface: clipping, and most of the mesh outside the view
        _frame("closeup", 200000, 1920, 1080, "normalmap", shadow=-1, dist=1.12, tex=1024),
        # many small scenes in one launch sequence
        {"name": "batch_small", "family": "batch", "scenes": 32, "tri_lo": 1000, "tri_hi": 20000,
         "px_lo": 128 * 128, "px_hi": 384 * 384, "tex": 256},
        # the benchmark's batched scenes (1k-200k triangles, 128^2-1024^2 pixels)
        {"name": "batch", "family": "batch", "scenes": 64, "tri_lo": 1000, "tri_hi": 200000,
         "px_lo": 128 * 128, "px_hi": 1024 * 1024, "tex": 512},
        # a burst of requests over resident meshes (5k-500k triangles, 256^2-1920x1080)
        {"name": "serve", "family": "serve", "scenes": 24, "meshes": 8, "tri_lo": 5000, "tri_hi": 500000,
         "px_lo": 256 * 256, "px_hi": 1920 * 1080, "tex": 512},
        # the micro-triangle frame: 20 M triangles at 3840x2160
        {"name": "micro", "family": "micro", "layers": 8, "grid": 1119, "width": 3840, "height": 2160,
         "shadow": 4096, "fp32": False, "tex": 2048},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi):
    """A pixel count, log-uniform, at an aspect between 1/2 and 2."""
    px, aspect = _log(rng, lo, hi), _log(rng, 0.5, 2.0)
    return max(16, round(math.sqrt(px * aspect))), max(16, round(math.sqrt(px / aspect)))


def draw(rng):
    family = rng.choice(["frame", "frame", "frame", "viewer", "models", "batch", "serve", "micro"])
    tex = rng.choice([256, 512, 1000, 1024])
    if family in ("frame", "viewer"):
        w, h = _size(rng, 128 * 128, 3840 * 2160 if family == "frame" else 1920 * 1080)
        c = _frame("", round(_log(rng, 12, 1.3e6 if family == "frame" else 2e5)), w, h, rng.choice(sorted(SHADERS)),
                   shadow=rng.choice([0, 0, -1, 1024, 2048, 1531]), fp32=rng.random() < 0.25,
                   objects=rng.randint(1, 8), dist=round(rng.uniform(1.1, 3.0), 3), tex=tex, family=family)
        c.pop("name")
        return c
    if family == "models":
        w, h = _size(rng, 256 * 256, 1920 * 1080)
        return {"family": family, "tris": round(_log(rng, 1e3, 3e5)), "objects": rng.randint(2, 24), "width": w,
                "height": h, "tex": tex}
    if family in ("batch", "serve"):
        lo, plo = round(_log(rng, 500, 5000)), round(_log(rng, 100 * 100, 300 * 300))
        c = {"family": family, "scenes": rng.randint(5, 64), "tri_lo": lo, "tri_hi": round(_log(rng, lo, 2e5)),
             "px_lo": plo, "px_hi": round(_log(rng, plo, 1024 * 1024)), "tex": rng.choice([256, 512])}
        return dict(c, scenes=rng.randint(3, 32), meshes=rng.randint(2, 8)) if family == "serve" else c
    w, h = _size(rng, 640 * 480, 3840 * 2160)
    return {"family": family, "layers": rng.randint(1, 8), "grid": round(_log(rng, 200, 1100)), "width": w, "height": h,
            "shadow": rng.choice([0, 1024, 2048, 4001]), "fp32": rng.random() < 0.25, "tex": tex}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _grid_edge(tris):
    """An object is six n x n grids: 12 n^2 triangles."""
    return max(1, round(math.sqrt(tris / 12.0)))


def _blob(rng, n, box):
    """A cube of n x n grids per side, or that cube inflated to a displaced sphere."""
    g = np.linspace(-1.0, 1.0, n + 1)
    a, b = np.meshgrid(g, g, indexing="ij")
    wave, phase = rng.uniform(1.5, 5.0, (4, 3)), rng.uniform(0, 2 * np.pi, 4)
    q = np.arange((n + 1) ** 2, dtype=np.int32).reshape(n + 1, n + 1)
    quad = np.stack([q[:-1, :-1], q[1:, :-1], q[:-1, 1:], q[1:, :-1], q[1:, 1:], q[:-1, 1:]], -1).reshape(-1, 3)
    pos, nrm, uv, idx = [], [], [], []
    for axis in range(3):
        for side in (-1.0, 1.0):
            p = np.empty((n + 1, n + 1, 3))
            p[..., axis], p[..., (axis + 1) % 3], p[..., (axis + 2) % 3] = side, a, b
            if not box:
                p /= np.linalg.norm(p, axis=-1, keepdims=True)
                p *= 1.0 + 0.0125 * sum(np.sin(p @ w + f) for w, f in zip(wave, phase))[..., None]
            m = np.cross(np.gradient(p, axis=0), np.gradient(p, axis=1)) * side
            pos.append(p.reshape(-1, 3))
            nrm.append((m / np.linalg.norm(m, axis=-1, keepdims=True)).reshape(-1, 3))
            uv.append(np.stack([(a + 1) / 2, (b + 1) / 2], -1).reshape(-1, 2))
            idx.append((quad if side > 0 else quad[:, ::-1]) + len(idx) * (n + 1) ** 2)
    return sg.Mesh(np.concatenate(pos).astype(np.float32), np.concatenate(nrm).astype(np.float32),
                   sg.clamp_uv(np.concatenate(uv)), np.ascontiguousarray(np.concatenate(idx), np.int32))


def _mesh(rng, tris, objects):
    """One displaced sphere, or several spheres and boxes placed around the origin."""
    parts = []
    for k in range(objects):
        m = _blob(rng, _grid_edge(tris / objects), objects > 1 and k % 2 == 1)
        rot = sg.rotation_matrix(rng).astype(np.float32)
        scale, off = (1.0, 0.0) if objects == 1 else (rng.uniform(0.18, 0.45), rng.uniform(-0.55, 0.55, 3))
        parts.append(sg.Mesh((m.pos @ rot.T * np.float32(scale) + off).astype(np.float32), m.nrm @ rot.T, m.uv, m.idx))
    return sg.merge(parts)


def _noise(rng, size, channels):
    """Value noise of four octaves: (size, size, channels) in [0, 1]."""
    acc = 0.0
    for octave in range(4):
        cells = torch.from_numpy(rng.random((1, channels, 8 << octave, 8 << octave), np.float32))
        acc = acc + F.interpolate(cells, size=(size, size), mode="bilinear", align_corners=True) * 0.5 ** octave
    return (acc / 1.875)[0].permute(1, 2, 0).contiguous().numpy()


def _diffuse(rng, size):
    img = np.full((size, size, 4), 255, np.uint8)
    img[..., :3] = (40 + 200 * _noise(rng, size, 3)).astype(np.uint8)
    return img


def _normal(rng, size):
    """A tangent-space normal map of a noisy height field, bytes B, G, R, A = z, y, x, 255."""
    h = _noise(rng, size, 1)[..., 0] * (0.06 * size)
    dy, dx = np.gradient(h)
    inv = 1.0 / np.sqrt(dx * dx + dy * dy + 1.0)
    img = np.full((size, size, 4), 255, np.uint8)
    for k, c in enumerate((inv, -dy * inv, -dx * inv)):
        img[..., k] = (c * 127.5 + 127.5).astype(np.uint8)
    return img


def _micro_mesh(rng, case):
    """Jittered grids that face the camera at (0, 0, 2) and fill the view, in
    pairs of equal positions (depth ties) at different uvs."""
    n = case["grid"]
    g = np.arange(n, dtype=np.float32) / np.float32(n - 1)
    q = np.arange(n * n, dtype=np.int32).reshape(n, n)
    quad = np.stack([q[:-1, :-1], q[:-1, 1:], q[1:, :-1], q[:-1, 1:], q[1:, 1:], q[1:, :-1]], -1).reshape(-1, 3)
    pos, uv, idx = [], [], []
    for layer in range(case["layers"]):
        if layer % 2 == 0:
            z = rng.uniform(-0.6, 0.6)
            half_h = (2.0 - z) * math.tan(math.radians(30.0)) * 1.02
            half_w = half_h * case["width"] / case["height"]
            jit = rng.random((n, n, 2), np.float32) * np.float32(0.6 / (n - 1)) - np.float32(0.3 / (n - 1))
            p = np.empty((n, n, 3), np.float32)
            p[..., 0] = ((g[None, :] + jit[..., 0]) * 2 - 1) * np.float32(half_w)
            p[..., 1] = ((g[:, None] + jit[..., 1]) * 2 - 1) * np.float32(half_h)
            p[..., 2] = z
        shift = rng.uniform(0, 0.5, 2).astype(np.float32)
        t = np.empty((n, n, 2), np.float32)
        t[..., 0], t[..., 1] = g[None, :] * np.float32(0.49) + shift[0], g[:, None] * np.float32(0.49) + shift[1]
        pos.append(p.reshape(-1, 3))
        uv.append(t.reshape(-1, 2))
        idx.append(quad + layer * n * n)
    pos = np.concatenate(pos)
    nrm = np.zeros_like(pos)
    nrm[:, 2] = 1.0
    return sg.Mesh(pos, nrm, np.concatenate(uv), np.concatenate(idx))


# ---------------------------------------------------------------------------
# what a program holds
# ---------------------------------------------------------------------------

_HELD = {}


def _context():
    """The program's one context, for the life of the process."""
    if "ctx" not in _HELD:
        _HELD["ctx"] = gpu.Context(0)
    return _HELD["ctx"]


def _server():
    if "server" not in _HELD:
        _HELD["server"] = gpu.Server(_context(), lanes=3)
    return _HELD["server"]


class _Owned:
    """A mesh, texture or target of the context, destroyed with the last that uses it."""

    def __init__(self, ctx, kind, handle):
        self.ctx, self.kind, self.handle = ctx, kind, handle

    def __del__(self):
        getattr(self.ctx.lib, "hana_%s_destroy" % self.kind)(self.ctx.h, self.handle)


class _TargetWords(ctypes.Structure):
    """How a target handle begins: its size, then its colour and depth planes."""
    _fields_ = [("width", ctypes.c_int32), ("height", ctypes.c_int32), ("color", ctypes.c_void_p),
                ("depth", ctypes.c_void_p)]


class _Plane:
    def __init__(self, owner, address, shape, typestr):
        self.owner = owner   # a tensor over the plane holds on to its target
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (address, False), "version": 2}


def _planes(target, width, height):
    """A resident target's colour bytes and depth words as tensors, without a
    copy: the images of a program that goes on with them on the GPU."""
    t = _TargetWords.from_address(target.handle.value)
    if (t.width, t.height) != (width, height):
        raise RuntimeError("a target handle no longer begins with its size")
    return [torch.as_tensor(_Plane(target, t.color, (height, width, 4), "|u1"), device="cuda"),
            torch.as_tensor(_Plane(target, t.depth, (height, width), "<i4"), device="cuda")]


class _State:
    """The resident objects of one case, given back with it."""

    def __init__(self, case, seed):
        self.case, self.ctx, self.owned, self.batch = case, _context(), [], None
        self.rng = np.random.default_rng(seed)

    def keep(self, kind, handle):
        self.owned.append(_Owned(self.ctx, kind, handle))
        return handle

    def mesh(self, m):
        return self.keep("mesh", self.ctx.mesh(m))

    def texture(self, img):
        return self.keep("texture", self.ctx.texture(img))

    def target(self, w, h):
        return self.keep("target", self.ctx.target(w, h))

    def image(self, w, h):
        """A target, and its planes as tensors."""
        handle = self.target(w, h)
        return handle, _planes(self.owned[-1], w, h)

    def material(self, shader, tex):
        return (self.texture(_diffuse(self.rng, tex)) if shader in DIFFUSE else None,
                self.texture(_normal(self.rng, tex)) if shader == "normalmap" else None)

    def __del__(self):
        if self.batch is not None:
            self.batch.close()


def _uniforms(rng, width, height, shadow, fp32, dist, front=False):
    cam = (0.0, 0.0, 2.0) if front else sg.orbit_camera(rng, dist, dist)
    scene = sg.Scene(None, width, height, sg.BLINN, shadow, cam, sg.random_light(rng, front=front), None, None,
                     shadow_fp32=fp32)
    return gpu.build_uniforms(scene)


def _shadow_size(case):
    s = case["shadow"]
    return None if s == 0 else (case["width"], case["height"]) if s < 0 else (s, s)


def _spread(case):
    """The sizes of a batch's or burst's scenes: triangle counts and pixel
    counts over their ranges, paired by a fixed shuffle, shaders and shadows in
    turn."""
    n = case["scenes"]
    at = (np.arange(n) + 0.5) / n
    mix = np.random.default_rng(n).permutation(n)
    tris = case["tri_lo"] * (case["tri_hi"] / case["tri_lo"]) ** at
    px = case["px_lo"] * (case["px_hi"] / case["px_lo"]) ** at[mix]
    aspect = 0.5 * 4.0 ** at[mix[::-1]]
    return [{"tris": int(t), "width": max(16, round(math.sqrt(p * a))), "height": max(16, round(math.sqrt(p / a))),
             "shader": "blinn" if k % 2 else "normalmap", "shadow": -1 if k % 4 < 2 else 0, "fp32": False,
             "objects": 1 + k % 8, "tex": case["tex"]} for k, (t, p, a) in enumerate(zip(tris, px, aspect))]


def prepare(case, seed):
    st = _State(case, seed)
    rng, ctx, family = st.rng, st.ctx, case["family"]
    if family in ("frame", "viewer", "micro"):
        micro = family == "micro"
        shader = "normalmap" if micro else case["shader"]
        size = _shadow_size(case)
        mesh = st.mesh(_micro_mesh(rng, case) if micro else _mesh(rng, case["tris"], case["objects"]))
        diffuse, normal = st.material(shader, case["tex"])
        u = _uniforms(rng, case["width"], case["height"], size is not None, case["fp32"], case.get("dist"), front=micro)
        st.screen, st.out = st.image(case["width"], case["height"])
        shadow_map = st.target(*size) if size else None
        st.frame = (mesh, SHADERS[shader], size is not None, u, st.screen, shadow_map, diffuse, normal)
    elif family == "models":
        st.screen, st.out = st.image(case["width"], case["height"])
        st.models = []
        eye, light = sg.orbit_camera(rng, 2.2, 2.2), sg.random_light(rng)
        for k in range(case["objects"]):
            shader = MODEL_SHADERS[k % len(MODEL_SHADERS)]
            # the models share the eye and the light; each has its place in the room
            scene = sg.Scene(None, case["width"], case["height"], SHADERS[shader], False, eye, light, None, None,
                             obj_position=tuple(rng.uniform(-0.6, 0.6, 3)), obj_rotation=tuple(rng.uniform(-180, 180, 3)),
                             obj_scale=(0.35, 0.35, 0.35))
            mesh = st.mesh(_blob(rng, _grid_edge(case["tris"] / case["objects"]), k % 3 == 2))
            st.models.append((mesh, SHADERS[shader], gpu.build_uniforms(scene), st.screen) + st.material(shader, case["tex"]))
    elif family == "batch":
        st.batch = gpu.Batch(ctx)
        material = st.material("normalmap", case["tex"])
        st.images = []
        for s in _spread(case):
            size = _shadow_size(s)
            mesh = st.mesh(_mesh(rng, s["tris"], s["objects"]))
            target, planes = st.image(s["width"], s["height"])
            u = _uniforms(rng, s["width"], s["height"], size is not None, False, 2.4)
            st.batch.add(ctx.frame_desc(mesh, SHADERS[s["shader"]], size is not None, u, target,
                                        st.target(*size) if size else None, *material))
            st.images.append(planes)
        st.batch.finalize(use_graph=True)
    else:
        material = st.material("normalmap", case["tex"])
        st.server = _server()
        tris = np.geomspace(case["tri_lo"], case["tri_hi"], case["meshes"])
        meshes = [st.mesh(_mesh(rng, t, 1)) for t in tris]
        st.requests = [(meshes[k % len(meshes)], SHADERS[s["shader"]], s["shadow"] != 0, s["width"], s["height"],
                        sg.orbit_camera(rng, 2.2, 3.2), sg.random_light(rng)) + material
                       for k, s in enumerate(_spread(case))]
    return st


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------

def run(st):
    ctx, family = st.ctx, st.case["family"]
    if family == "batch":
        st.batch.run()
        # 64 images at most come back; of up to 32 scenes their depth too
        return [p if len(st.images) <= 32 else p[0] for p in st.images]
    if family == "serve":
        for tag, request in enumerate(st.requests):
            st.server.submit(*request, tag=tag)
        images = [None] * len(st.requests)
        left = len(images)
        while left:
            for c in st.server.poll(256, wait_ms=50):
                if c.status != 0:
                    raise RuntimeError("a request failed: %d" % c.status)
                images[int(c.user_tag)] = st.server.image(c)
                st.server.release(int(c.id))
                left -= 1
        return images
    ctx.clear(st.screen)
    if family == "models":
        for mesh, shader, u, screen, diffuse, normal in st.models:
            ctx.draw(mesh, shader, u, screen, diffuse, normal)
        return st.out
    ctx.render_frame(*st.frame)
    if family == "viewer":
        return ctx.present(st.screen, st.case["width"], st.case["height"])
    return st.out


# ---------------------------------------------------------------------------
# the work
# ---------------------------------------------------------------------------

def _frame_work(verts, tris, width, height, shadow, fp32, texels):
    """Each pass reads 32 B a vertex and 12 B a face; colour and depth are
    written once, a shadow map written (its depth alone with fp32) and sampled
    once, each texel read once.  A vertex takes a 4x4 product (28 operations)
    per pass, a face its cross product (9), a pixel one depth comparison."""
    passes = 2 if shadow else 1
    px, spx = width * height, shadow[0] * shadow[1] if shadow else 0
    return np.array([passes * (verts * 32 + tris * 12) + px * 8 + spx * ((4 if fp32 else 8) + 4) + texels * 4,
                     passes * (verts * 28 + tris * 9) + px + spx], float)


def _mesh_counts(tris, objects):
    n = _grid_edge(tris / objects)
    return objects * 6 * (n + 1) ** 2, objects * 12 * n * n


def _texels(shader, tex):
    return ((shader in DIFFUSE) + (shader == "normalmap")) * tex * tex


def work(case):
    family = case["family"]
    if family == "micro":
        n, k = case["grid"], case["layers"]
        total = _frame_work(k * n * n, k * 2 * (n - 1) ** 2, case["width"], case["height"], _shadow_size(case),
                            case["fp32"], 2 * case["tex"] ** 2)
    elif family in ("frame", "viewer"):
        total = _frame_work(*_mesh_counts(case["tris"], case["objects"]), case["width"], case["height"],
                            _shadow_size(case), case["fp32"], _texels(case["shader"], case["tex"]))
        if family == "viewer":
            total[0] += case["width"] * case["height"] * 8   # read again, the image written
    elif family == "models":
        total = np.array([case["width"] * case["height"] * 8.0, 0.0])
        for k in range(case["objects"]):
            v, t = _mesh_counts(case["tris"] / case["objects"], 1)
            total += _frame_work(v, t, 0, 0, None, False, _texels(MODEL_SHADERS[k % len(MODEL_SHADERS)], case["tex"]))
    else:
        sizes = _spread(case)
        tris = np.geomspace(case["tri_lo"], case["tri_hi"], case["meshes"]) if family == "serve" else None
        total = np.array([2.0 * 4 * case["tex"] ** 2, 0.0])
        for k, s in enumerate(sizes):
            counts = _mesh_counts(s["tris"], s["objects"]) if tris is None else _mesh_counts(tris[k % len(tris)], 1)
            total += _frame_work(*counts, s["width"], s["height"], _shadow_size(s), False, 0)
            if family == "serve":
                total[0] += s["width"] * s["height"] * 4     # the image on the host
    return {"bytes": float(total[0]), "flops": float(total[1])}
