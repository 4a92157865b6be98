"""Scenes whose triangles the chunked binning has no room for, by their order or
by how they crowd: counted binning renders them, against the oracle (depth
bit-exact, colour as in test_gpu_parity)."""
import ctypes as C

import numpy as np
import pytest

from hana_amd import scenegen as sg
from parity import assert_color_ok, assert_depth_exact
from pyoracle import CPURenderer, HostTarget
from test_gpu_parity import soup_scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oracle():
    return CPURenderer("oracle")


def layered_scene(layers, nx, ny, width, height, seed, kind=sg.TEXTURE, fill=0.98, order="random"):
    """Planes of nx x ny quads that fill the view from (0, 0, 2), one behind the
    other, jittered, with their faces in random order or row by row."""
    rng = np.random.default_rng(seed)
    gx, gy = np.meshgrid(np.linspace(-1, 1, nx + 1), np.linspace(-1, 1, ny + 1))
    q = np.arange((nx + 1) * (ny + 1), dtype=np.int32).reshape(ny + 1, nx + 1)
    quad = np.stack([q[:-1, :-1], q[:-1, 1:], q[1:, :-1], q[:-1, 1:], q[1:, 1:], q[1:, :-1]], -1).reshape(-1, 3)
    pos, idx = [], []
    for k in range(layers):
        z = 0.5 - k / layers
        half = (2.0 - z) * np.tan(np.radians(30.0)) * fill
        jit = rng.uniform(-0.3, 0.3, (2,) + gx.shape)
        pos.append(np.stack([(gx + jit[0] * 2 / nx * (np.abs(gx) < 1)) * half * width / height,
                             (gy + jit[1] * 2 / ny * (np.abs(gy) < 1)) * half, np.full_like(gx, z)], -1).reshape(-1, 3))
        idx.append(quad + k * q.size)
    pos, idx = np.concatenate(pos).astype(np.float32), np.concatenate(idx)
    if order == "random":
        idx = idx[rng.permutation(len(idx))]
    nrm = np.zeros_like(pos)
    nrm[:, 2] = 1.0
    uv = np.tile(np.stack([(gx + 1) / 2, (gy + 1) / 2], -1).reshape(-1, 2), (layers, 1))
    base = sg.small_scene(kind, width=width, height=height, seed=seed)
    mesh = sg.Mesh(pos, nrm, sg.clamp_uv(uv), np.ascontiguousarray(idx, np.int32))
    return sg.Scene(mesh, width, height, kind, False, (0.0, 0.0, 2.0), base.light_pos, base.diffuse, base.normal,
                    name=f"{layers} layers")


def oracle_image(oracle, scene):
    ref = HostTarget(scene.width, scene.height)
    oracle.draw(scene.mesh, scene.shader, oracle.build_uniforms(scene), ref, scene.diffuse, scene.normal)
    return ref


# layers and quads of a layer: 1,747,200 faces, just under the most that the
# fixed workspace admits at this size (1.8 M), with three tiles each; crowded
# into few tiles, with triangles of more than 16 tiles between
NOALLOC = {
    "most-faces": lambda: layered_scene(70, 160, 78, 1920, 1080, 5),
    "crowded": lambda: layered_scene(300, 20, 20, 1920, 1080, 6, kind=sg.BLINN, fill=0.08),
    "wide-between": lambda: sg_merge(layered_scene(250, 24, 24, 1280, 720, 7, fill=0.1), soup_scene(900, 1280, 720, 100, 200, 8)),
}


def sg_merge(a, b):
    return sg.Scene(sg.merge([a.mesh, b.mesh]), a.width, a.height, a.shader, False, a.cam_pos, a.light_pos, a.diffuse,
                    a.normal, name=a.name)


@pytest.mark.parametrize("tile,wgs", [(16, 0), (32, 2)])
@pytest.mark.parametrize("name", NOALLOC)
def test_noalloc_whatever_the_order(oracle, name, tile, wgs):
    """A frame that the fixed workspace admits is rendered whatever the order of
    its faces, as often as it is called, and so is the one after it."""
    from hana_amd.gpu import Context, build_uniforms
    scene = NOALLOC[name]()
    plain = soup_scene(3000, 320, 200, 2, 30, 9)
    with Context(0) as ctx:
        ctx.set_tuning(tile, wgs)
        images = []
        for s in (scene, plain):
            t = ctx.target(s.width, s.height)
            images.append((s, t, ctx.frame_desc(ctx.mesh(s.mesh), s.shader, False, build_uniforms(s), t, None,
                                                ctx.texture(s.diffuse), ctx.texture(s.normal))))
        ctx.sync()
        for _, _, d in images + images:
            ctx.check(ctx.lib.hana_render_frame_noalloc(ctx.h, C.byref(d)), "noalloc")
        for s, t, _ in images:
            col, dep = ctx.read(t, s.width, s.height)
            ref = oracle_image(oracle, s)
            assert_depth_exact(dep, ref.depth, s.name)
            assert_color_ok(col, ref.color, s.name)
