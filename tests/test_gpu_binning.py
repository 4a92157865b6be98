"""The GPU's binning at the sizes where its paths change, against the oracle:
depth and the winning face of every pixel bit-exact, colour as in
test_gpu_parity."""
import ctypes as C

import numpy as np
import pytest

from hana_amd import scenegen as sg
from parity import assert_color_ok, assert_depth_exact
from pyoracle import CPURenderer, HostTarget
from test_gpu_parity import check_scene, soup_scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from hana_amd.gpu import Context
    c = Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def oracle():
    return CPURenderer("oracle")


# faces, target, triangle size in pixels, spread (> 1: part of the faces is clipped)
CASES = {
    "one-face": (1, (64, 64), (20, 40), 1.0),
    # a workgroup of the one-launch geometry holds 256 faces
    "front-255": (255, (320, 240), (4, 12), 1.0),
    "front-257": (257, (320, 240), (4, 12), 1.0),
    # more distinct tiles in a workgroup than its table has slots
    "front-scattered": (700, (1900, 1070), (40, 60), 1.0),
    "front-clipped": (1500, (333, 222), (10, 60), 1.6),
    # one launch up to 2^18 faces, then vertex, set-up and clip launches
    "front-largest": (1 << 18, (640, 480), (1, 4), 1.3),
    "staged-smallest": ((1 << 18) + 1, (640, 480), (1, 4), 1.3),
    "staged-remainder": ((1 << 18) + 1023, (640, 480), (1, 4), 1.0),
    # triangles of more than 16 tiles go to the pass's list of 512, then into
    # the tiles' own lists
    "wide-512": (512, (640, 480), (150, 220), 1.0),
    "wide-700": (700, (640, 480), (150, 220), 1.2),
    "wide-long": (3, (8000, 48), (12000, 16000), 1.0),
    # crowded into few tiles: more descriptors than a tile has places, in the
    # list behind them; past that list, with more places in every tile; on a
    # target of so many tiles that only the list grows
    "crowded-list": (60_000, (2048, 1024), (100, 400), 0.01),
    "crowded-places": (120_000, (2048, 1024), (100, 400), 0.01),
    "crowded-large": (140_000, (4096, 4096), (100, 400), 0.01),
    # 32x32 tiles from 8,000 16x16 tiles and 128 pixels per face on
    "tiles-16": (16_257, (1930, 1078), (4, 30), 1.0),
    "tiles-32": (16_253, (1930, 1078), (4, 30), 1.0),
    "tiles-32-clipped": (3000, (2049, 1025), (30, 90), 1.5),
    # two waves per raster workgroup from 10,000 16x16 tiles and 4 pixels per face on
    "waves-4-tiles": (30_000, (1584, 1600), (4, 30), 1.0),
    "waves-2": (30_000, (1599, 1600), (4, 30), 1.0),
    "waves-2-clipped": (200_000, (1600, 1600), (2, 9), 1.3),
    "waves-4-faces": (640_001, (1600, 1600), (1, 4), 1.0),
}


@pytest.mark.parametrize("name", CASES)
def test_binning_paths(ctx, oracle, name):
    n, wh, px, spread = CASES[name]
    scene = soup_scene(n, wh[0], wh[1], px[0], px[1], seed=500 + n)
    scene.mesh.pos[:, :2] *= np.float32(spread)
    check_scene(ctx, oracle, scene)


@pytest.mark.parametrize("faces", [(300, 33_000), (33_000, 300)])
def test_calls_on_one_target_keep_order(ctx, oracle, faces):
    """Calls of few faces draw on the slot of their target, larger ones on the
    next: eight calls that alternate between the two and between two targets,
    one of them a shadow map of the other's shadowed draws, give the frames of
    the calls in their order."""
    from hana_amd.gpu import SHADOW, build_uniforms
    scenes = [soup_scene(f, 160, 120, 2, 24, seed=40 + i) for i, f in enumerate(faces * 2)]
    for s in scenes:
        s.shadow = True
    big, smap = ctx.target(160, 120), ctx.target(160, 120)
    o_big, o_smap = HostTarget(160, 120), HostTarget(160, 120)
    for s in scenes:
        args = (ctx.mesh(s.mesh), ctx.texture(s.diffuse), ctx.texture(s.normal))
        ctx.draw(args[0], SHADOW, build_uniforms(s), smap, args[1], args[2])
        ctx.draw(args[0], s.shader, build_uniforms(s), big, args[1], args[2], smap)
        u = oracle.build_uniforms(s)
        oracle.draw(s.mesh, sg.SHADOW, u, o_smap, s.diffuse, s.normal)
        oracle.draw(s.mesh, s.shader, u, o_big, s.diffuse, s.normal, o_smap)
    col, dep = ctx.read(big, 160, 120)
    assert_depth_exact(dep, o_big.depth, "target")
    assert_color_ok(col, o_big.color, "target")
    assert_depth_exact(ctx.read(smap, 160, 120)[1], o_smap.depth, "shadow map")


@pytest.mark.parametrize("name", ["crowded-places", "wide-700", "front-scattered", "front-clipped"])
def test_binning_in_fixed_scratch(ctx, oracle, name):
    """The frame without allocation bins into a workspace of fixed size, with
    every wide triangle listed and its own list behind the tiles' places."""
    from hana_amd.gpu import build_uniforms
    n, (w, h), px, spread = CASES[name]
    scene = soup_scene(n, w, h, px[0], px[1], seed=700 + n)
    scene.mesh.pos[:, :2] *= np.float32(spread)
    target = ctx.target(w, h)
    desc = ctx.frame_desc(ctx.mesh(scene.mesh), scene.shader, False, build_uniforms(scene), target, None,
                          ctx.texture(scene.diffuse), ctx.texture(scene.normal))
    ctx.sync()
    ctx.check(ctx.lib.hana_render_frame_noalloc(ctx.h, C.byref(desc)), "noalloc")
    col, dep = ctx.read(target, w, h)
    ref = HostTarget(w, h)
    oracle.draw(scene.mesh, scene.shader, oracle.build_uniforms(scene), ref, scene.diffuse, scene.normal)
    assert_depth_exact(dep, ref.depth, name)
    assert_color_ok(col, ref.color, name)


@pytest.mark.parametrize("edge,parts", [(1040, 1), (1056, 2), (3568, 2), (3584, 4)])
def test_batch_parts_by_tiles(ctx, edge, parts):
    """Four frames of edge x edge: one part up to 17,000 16x16 tiles, two up to
    200,000, four beyond; each with the images of the frames drawn one by one."""
    from hana_amd.gpu import Batch, build_uniforms
    batch, frames = Batch(ctx), []
    for k in range(4):
        s = soup_scene(200 + 100 * k, edge, edge, 10, 60, seed=800 + k)
        u, mesh = build_uniforms(s), ctx.mesh(s.mesh)
        tex = (ctx.texture(s.diffuse), ctx.texture(s.normal))
        t, single = ctx.target(edge, edge), ctx.target(edge, edge)
        batch.add(ctx.frame_desc(mesh, s.shader, False, u, t, None, *tex))
        ctx.draw(mesh, s.shader, u, single, *tex)
        frames.append((t, single))
    batch.finalize(use_graph=True)
    assert batch.tuning()["parts"] == parts
    batch.run()
    for t, single in frames:
        got, want = ctx.read(t, edge, edge), ctx.read(single, edge, edge)
        assert np.array_equal(got[0], want[0]) and got[1].tobytes() == want[1].tobytes()
    batch.close()


@pytest.mark.parametrize("faces", [3 << 17, (3 << 17) + 1])
def test_batch_part_at_the_one_launch_limit(ctx, faces):
    """A batch's part of up to 3 x 2^17 faces runs its geometry in one launch,
    a larger one in three: both render what the single draw does."""
    from hana_amd.gpu import Batch, build_uniforms
    s = soup_scene(faces, 640, 480, 1, 4, seed=900)
    s.mesh.pos[:, :2] *= np.float32(1.2)
    u, mesh, tex = build_uniforms(s), ctx.mesh(s.mesh), (ctx.texture(s.diffuse), ctx.texture(s.normal))
    t, single = ctx.target(640, 480), ctx.target(640, 480)
    batch = Batch(ctx)
    batch.add(ctx.frame_desc(mesh, s.shader, False, u, t, None, *tex))
    batch.finalize(use_graph=True)
    ctx.draw(mesh, s.shader, u, single, *tex)
    batch.run()
    got, want = ctx.read(t, 640, 480), ctx.read(single, 640, 480)
    assert np.array_equal(got[0], want[0]) and got[1].tobytes() == want[1].tobytes()
    batch.close()
