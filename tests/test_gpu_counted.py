"""Scenes whose triangles the chunked binning has no room for, by their order or
by how they crowd: counted binning renders them, against the oracle (depth
bit-exact, colour as in test_gpu_parity)."""
import ctypes as C
import dataclasses
import time

import numpy as np
import pytest

from hana_amd import scenegen as sg
from parity import assert_color_ok, assert_depth_exact
from pyoracle import CPURenderer, HostTarget
from test_gpu_parity import soup_scene, straddling_scene
from test_gpu_serve import collect

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def oracle():
    return CPURenderer("oracle")


def layered_scene(layers, nx, ny, width, height, seed, kind=sg.TEXTURE, fill=0.98, jitter=0.3):
    """Planes of nx x ny quads that fill the view from (0, 0, 2), one behind the
    other, jittered, with their faces in random order."""
    rng = np.random.default_rng(seed)
    gx, gy = np.meshgrid(np.linspace(-1, 1, nx + 1), np.linspace(-1, 1, ny + 1))
    q = np.arange((nx + 1) * (ny + 1), dtype=np.int32).reshape(ny + 1, nx + 1)
    quad = np.stack([q[:-1, :-1], q[:-1, 1:], q[1:, :-1], q[:-1, 1:], q[1:, 1:], q[1:, :-1]], -1).reshape(-1, 3)
    pos, idx = [], []
    for k in range(layers):
        z = 0.5 - k / layers
        half = (2.0 - z) * np.tan(np.radians(30.0)) * fill
        jit = rng.uniform(-jitter, jitter, (2,) + gx.shape)
        pos.append(np.stack([(gx + jit[0] * 2 / nx * (np.abs(gx) < 1)) * half * width / height,
                             (gy + jit[1] * 2 / ny * (np.abs(gy) < 1)) * half, np.full_like(gx, z)], -1).reshape(-1, 3))
        idx.append(quad + k * q.size)
    pos, idx = np.concatenate(pos).astype(np.float32), np.concatenate(idx)
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


def test_many_more_descriptors_than_places():
    """7.5 million triangles in random order, of 9 to 16 tiles each: 95 million
    descriptors, where a workspace has places for 16 million at first.  The draw gives the
    image that its faces give in eight draws, in their order; so does a batch,
    and neither needs rendering again from then on."""
    from hana_amd.gpu import Batch, Context, build_uniforms
    scene = layered_scene(3720, 42, 24, 1920, 1080, 11, fill=1.008, jitter=0.0)
    mesh = scene.mesh
    with Context(0) as ctx:
        u = build_uniforms(scene)
        tex = (ctx.texture(scene.diffuse), ctx.texture(scene.normal))
        whole, parts, batched = (ctx.target(1920, 1080) for _ in range(3))
        m = ctx.mesh(mesh)
        ctx.draw(m, scene.shader, u, whole, *tex)
        got = [ctx.read(whole, 1920, 1080)]
        replays = ctx.replay_count()
        for k in range(2):
            ctx.clear(whole)
            ctx.draw(m, scene.shader, u, whole, *tex)
            got.append(ctx.read(whole, 1920, 1080))
        assert ctx.replay_count() == replays
        batch = Batch(ctx)
        batch.add(ctx.frame_desc(m, scene.shader, False, u, batched, None, *tex))
        batch.finalize(use_graph=True)
        batch.run()
        batch.run()
        got.append(ctx.read(batched, 1920, 1080))
        batch.close()
    with Context(0) as ctx:
        tex = (ctx.texture(scene.diffuse), ctx.texture(scene.normal))
        parts = ctx.target(1920, 1080)
        for f in np.array_split(mesh.idx, 8):
            ctx.draw(ctx.mesh(sg.Mesh(mesh.pos, mesh.nrm, mesh.uv, np.ascontiguousarray(f))), scene.shader, u, parts, *tex)
            ctx.sync()
        col, dep = ctx.read(parts, 1920, 1080)
    assert (dep < 1e30).mean() > 0.99
    for c, d in got:
        assert d.tobytes() == dep.tobytes() and np.array_equal(c, col)


def test_more_descriptors_than_a_workspace_grows_to(oracle):
    """A quarter of a million triangles on a few dozen of 262,144 tiles: each of
    those has a descriptor of nearly every set-up workgroup, and as many places in
    every tile are more than a workspace grows to.  One overflow, then counted
    binning in each draw, whose shadow pass is binned so too; and in a batch."""
    from hana_amd.gpu import Batch, Context, build_uniforms
    scene = soup_scene(250_000, 8192, 8192, 100, 400, 13)
    scene.mesh.pos[:, :2] *= np.float32(0.01)
    ref = oracle_image(oracle, scene)
    with Context(0) as ctx:
        u, mesh = build_uniforms(scene), ctx.mesh(scene.mesh)
        tex = (ctx.texture(scene.diffuse), ctx.texture(scene.normal))
        t, frame, smap, batched = (ctx.target(8192, 8192) for _ in range(4))
        for k in range(2):
            ctx.clear(t)
            ctx.draw(mesh, scene.shader, u, t, *tex)
            col, dep = ctx.read(t, 8192, 8192)
            assert ctx.replay_count() == 1
            assert_depth_exact(dep, ref.depth, scene.name)
            assert_color_ok(col, ref.color, scene.name)
        ctx.render_frame(mesh, scene.shader, True, u, frame, smap, *tex)
        assert np.array_equal(ctx.read(frame, 8192, 8192)[1], dep)
        batch = Batch(ctx)
        batch.add(ctx.frame_desc(mesh, scene.shader, False, u, batched, None, *tex))
        batch.finalize(use_graph=True)
        for k in range(2):
            batch.run()
        got = ctx.read(batched, 8192, 8192)
        assert got[1].tobytes() == dep.tobytes() and np.array_equal(got[0], col)
        batch.close()


def frame_time(ctx, scene, frames=6):
    """The fastest of some frames, in seconds."""
    from hana_amd.gpu import build_uniforms
    args = (ctx.mesh(scene.mesh), scene.shader, build_uniforms(scene), ctx.target(scene.width, scene.height),
            ctx.texture(scene.diffuse), ctx.texture(scene.normal))
    best = 1e9
    for _ in range(frames):
        t0 = time.perf_counter()
        ctx.clear(args[3])
        ctx.draw(*args)
        ctx.sync()
        best = min(best, time.perf_counter() - t0)
    return best


def test_scattered_faces_take_no_longer_than_a_scan_of_their_entries():
    """Three million faces that crowd into a thousand tiles of a 4K target, in
    random order and row by row: a tile reads its own entries only, so the order
    costs a few times as much at most."""
    from hana_amd.gpu import Context
    scene = layered_scene(1, 1500, 1000, 3840, 2160, 14, fill=0.17, jitter=10.0)
    order = np.lexsort((np.arange(len(scene.mesh.idx)), scene.mesh.idx.min(1)))
    rows = sg.Mesh(scene.mesh.pos, scene.mesh.nrm, scene.mesh.uv, np.ascontiguousarray(scene.mesh.idx[order]))
    ordered = dataclasses.replace(scene, mesh=rows)
    with Context(0) as ctx:
        took = [frame_time(ctx, s) for s in (ordered, scene)]
    assert took[1] < 8 * took[0], took


def test_crowded_tile_takes_time_by_its_entries():
    """Sixteen times the triangles on the same two tiles take at most sixteen times
    as long (and a tenth for the clock): a list of a tile's entries begins where
    the one before ended."""
    from hana_amd.gpu import Context
    with Context(0) as ctx:
        took = []
        for n in (400_000, 6_400_000):
            scene = soup_scene(n, 1920, 1080, 500, 600, 15)
            scene.mesh.pos[:, :2] *= np.float32(0.005)
            took.append(frame_time(ctx, scene))
    assert took[1] < 17.6 * took[0], took


def test_counted_beside_an_overflow(oracle):
    """A server's batch that outgrew its lane's workspace is launched again with
    counted binning: frames of few and of many faces, of odd sizes, clipped, with
    triangles of one tile and of hundreds, with and without shadow maps."""
    from hana_amd.gpu import Context, Server
    scenes = [straddling_scene()]
    for k, (w, h, n) in enumerate([(65, 47, 1), (333, 217, 255), (1, 1, 40), (700, 900, 1025), (1930, 1078, 5000),
                                   (97, 61, 20_000), (640, 480, 700)]):
        s = soup_scene(n, w, h, *((100, 400) if n == 700 else (2, 90)), 60 + n)
        s.mesh.pos[:, :2] *= np.float32(1.2)
        s.shadow = k % 2 == 0
        scenes.append(s)
    first = soup_scene(1000, 3840, 2160, 2, 30, 3)
    with Context(0) as ctx:
        objects = [(ctx.mesh(s.mesh), ctx.texture(s.diffuse), ctx.texture(s.normal)) for s in [first] + scenes]
        # the first has a batch's pixels by itself; the others arrive while the
        # lane is busy with it, and are taken together
        server = Server(ctx, lanes=1, max_batch_frames=16, max_batch_pixels=8_000_000, return_depth=True)
        for k, (s, (m, d, n)) in enumerate(zip([first] + scenes, objects)):
            server.submit(m, s.shader, s.shadow, s.width, s.height, s.cam_pos, s.light_pos, d, n, tag=k)
        res = collect(server, 1 + len(scenes))
        st = server.stats()
        server.close()
    assert st["retries"] >= 1 and max(v[2] for v in res.values()) == len(scenes)
    for k, s in enumerate(scenes):
        status, img, _, dep = res[1 + k]
        ref, _, _ = oracle.render_frame(s)
        assert status == 0, s.name
        assert_depth_exact(dep, ref.depth, s.name)
        assert_color_ok(img, ref.color, s.name)


class MeshWords(C.Structure):
    """How a mesh handle begins: its counts, then its arrays on the device."""
    _fields_ = [("V", C.c_int32), ("F", C.c_int32), ("soa", C.c_void_p), ("idx", C.c_void_p)]


def move_vertices(ctx, mesh, pos):
    """Other positions for a resident mesh, as a program's own kernel would write them."""
    words = MeshWords.from_address(mesh.value)
    assert words.V == len(pos)
    xyz = np.ascontiguousarray(pos.T, np.float32)
    ctx.sync()
    assert ctx.lib.hipMemcpy(C.c_void_p(words.soa), xyz.ctypes.data_as(C.c_void_p), C.c_size_t(xyz.nbytes), C.c_int(1)) == 0


@pytest.mark.parametrize("parts,use_graph", [(1, True), (2, True), (3, False)])
def test_batch_outgrows_the_workspace_it_was_sized_for(parts, use_graph):
    """A part of a batch that needs more than its trial run did is run again,
    with the images of single draws: after one run and after several, with a
    draw or a clear of its targets behind it, and when it is destroyed."""
    from hana_amd.gpu import Batch, Context, build_uniforms
    scenes = [soup_scene(n, w, h, 100, 400, 70 + n) for n, w, h in ((900, 333, 217), (60_000, 2048, 1024), (300, 97, 61))]
    tops = [soup_scene(50, s.width, s.height, 20, 60, 80 + k) for k, s in enumerate(scenes)]
    spread = [s.mesh.pos.copy() for s in scenes]
    for s, p in zip(scenes, spread):
        p[:, :2] = s.mesh.pos.reshape(-1, 3, 3).mean(1, keepdims=True).repeat(3, 1).reshape(-1, 3)[:, :2]
        p[:, :2] += (s.mesh.pos[:, :2] - p[:, :2]) * np.float32(0.02)      # small triangles all over the view
        s.mesh.pos[:, :2] *= np.float32(0.03)                              # then in a few tiles
    with Context(0) as ctx:
        u = [build_uniforms(s) for s in scenes]
        tex = [(ctx.texture(s.diffuse), ctx.texture(s.normal)) for s in scenes]
        top = [ctx.mesh(s.mesh) for s in tops]
        want, topped = [], []
        for k, s in enumerate(scenes):
            t = ctx.target(s.width, s.height)
            ctx.draw(ctx.mesh(s.mesh), s.shader, u[k], t, *tex[k])
            want.append(ctx.read(t, s.width, s.height))
            ctx.draw(top[k], s.shader, u[k], t, *tex[k])
            topped.append(ctx.read(t, s.width, s.height))

        def same(targets, images, what):
            for t, s, (col, dep) in zip(targets, scenes, images):
                c, d = ctx.read(t, s.width, s.height)
                assert d.tobytes() == dep.tobytes() and np.array_equal(c, col), what

        for after in ("run", "runs", "draw", "clear", "destroy"):
            meshes = [ctx.mesh(sg.Mesh(p, s.mesh.nrm, s.mesh.uv, s.mesh.idx)) for p, s in zip(spread, scenes)]
            targets = [ctx.target(s.width, s.height) for s in scenes]
            batch = Batch(ctx)
            batch.set_tuning(16, 0, parts)
            for k, s in enumerate(scenes):
                batch.add(ctx.frame_desc(meshes[k], s.shader, False, u[k], targets[k], None, *tex[k]))
            batch.finalize(use_graph=use_graph)
            batch.run()
            for m, s in zip(meshes, scenes):
                move_vertices(ctx, m, s.mesh.pos)
            before = ctx.replay_count()
            for k in range(3 if after == "runs" else 1):
                batch.run()
            if after == "draw":
                for k, s in enumerate(scenes):
                    ctx.draw(top[k], s.shader, u[k], targets[k], *tex[k])
            elif after == "clear":
                ctx.clear(targets[1])
                col, dep = ctx.read(targets[1], 2048, 1024)
                assert (dep > 3e38).all() and not col[..., :3].any()
                targets, full = [targets[0], targets[2]], targets
            elif after == "destroy":
                batch.close()
            if after == "clear":
                for t, k in zip(targets, (0, 2)):
                    c, d = ctx.read(t, scenes[k].width, scenes[k].height)
                    assert d.tobytes() == want[k][1].tobytes() and np.array_equal(c, want[k][0])
                targets = full
            else:
                same(targets, topped if after == "draw" else want, after)
            assert ctx.replay_count() == before + 1
            if after != "destroy":
                batch.run()
                same(targets, want, "the run after")
                assert ctx.replay_count() == before + 1
                batch.close()


def test_batch_of_many_wide_triangles_renders_every_time():
    """More triangles of many tiles than a pass's list holds: which of them it
    holds differs from run to run, and the images do not."""
    from hana_amd.gpu import Batch, Context, build_uniforms
    scene = soup_scene(594, 640, 480, 500, 900, 90)
    with Context(0) as ctx:
        u, mesh, tex = build_uniforms(scene), ctx.mesh(scene.mesh), (ctx.texture(scene.diffuse), ctx.texture(scene.normal))
        single, t = ctx.target(640, 480), ctx.target(640, 480)
        ctx.draw(mesh, scene.shader, u, single, *tex)
        col, dep = ctx.read(single, 640, 480)
        batch = Batch(ctx)
        batch.add(ctx.frame_desc(mesh, scene.shader, False, u, t, None, *tex))
        batch.finalize(use_graph=True)
        junk = np.full((480, 640, 4), 0x5A, np.uint8), np.full((480, 640), 7, np.float32)
        for k in range(200):
            ctx.upload(t, *junk)
            batch.run()
            c, d = ctx.read(t, 640, 480)
            assert d.tobytes() == dep.tobytes() and np.array_equal(c, col), k
        batch.close()


@pytest.mark.parametrize("wh,shadow_wh,faces", [((1920, 1080), None, 5000), ((640, 480), (1024, 1024), 200_000)])
def test_server_budget_counts_the_workspace(wh, shadow_wh, faces):
    """A request is charged for its targets, its vertices' and faces' arrays and
    the tiles' chunk descriptors (8 bytes each)."""
    from hana_amd.gpu import Context, Server
    s = soup_scene(faces, *wh, 2, 30, 4)
    maps = [wh] + ([shadow_wh] if shadow_wh else [])
    tiles = sum(-(-w // 16) * -(-h // 16) for w, h in maps)
    per_tile = max(min(8 * (len(maps) * faces // tiles + 1), 512), 64) + 16
    least = sum(8 * w * h for w, h in maps) + len(maps) * (3 * faces * 49 + faces * 70) + tiles * 8 * per_tile
    with Context(0) as ctx:
        server = Server(ctx, lanes=1)
        server.submit(ctx.mesh(s.mesh), s.shader, shadow_wh is not None, *wh, s.cam_pos, s.light_pos, ctx.texture(s.diffuse),
                      ctx.texture(s.normal), shadow_wh=shadow_wh or (0, 0))
        res = collect(server, 1)
        st = server.stats()
        server.close()
    assert res[0][0] == 0 and least <= st["peak_inflight_bytes"] < 2 * least


def test_noalloc_frame_behind_a_batch_that_is_to_be_run_again():
    """A frame without allocation cannot be drawn again behind the batch: the wait
    says so, and the next run is right."""
    from hana_amd.gpu import HANA_E_OVERFLOW, Batch, Context, HanaError, build_uniforms
    scene = soup_scene(60_000, 2048, 1024, 2, 8, 91)
    crowded = scene.mesh.pos.copy()
    crowded[:, :2] *= np.float32(0.03)
    with Context(0) as ctx:
        u, tex = build_uniforms(scene), (ctx.texture(scene.diffuse), ctx.texture(scene.normal))
        mesh, t, other = ctx.mesh(scene.mesh), ctx.target(2048, 1024), ctx.target(2048, 1024)
        batch = Batch(ctx)
        batch.add(ctx.frame_desc(mesh, scene.shader, False, u, t, None, *tex))
        batch.finalize(use_graph=True)
        move_vertices(ctx, mesh, crowded)
        batch.run()
        d = ctx.frame_desc(mesh, scene.shader, False, u, other, None, *tex)
        ctx.check(ctx.lib.hana_render_frame_noalloc(ctx.h, C.byref(d)), "noalloc")
        with pytest.raises(HanaError) as err:
            ctx.sync()
        assert err.value.code == HANA_E_OVERFLOW and "no-alloc" in str(err.value)
        ctx.clear(other)
        ctx.draw(mesh, scene.shader, u, other, *tex)
        want = ctx.read(other, 2048, 1024)
        batch.run()
        got = ctx.read(t, 2048, 1024)
        assert got[1].tobytes() == want[1].tobytes() and np.array_equal(got[0], want[0])
        batch.close()
