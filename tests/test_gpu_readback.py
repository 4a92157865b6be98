"""Targets read back and presented: every byte, at the sizes where the way back
changes (bands of a plane, two planes in one staging buffer, pieces past it),
into memory that is warm, new, pinned, or not 16-byte aligned."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from hana_amd.gpu import Context
    c = Context(0)
    yield c
    c.close()


def _u8(a):
    return a.ctypes.data_as(C.POINTER(C.c_uint8))


def _f32(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


def _memory(ctx, kind, nbytes):
    if kind == "pinned":
        p = C.c_void_p()
        assert ctx.lib.hipHostMalloc(C.byref(p), C.c_size_t(nbytes), C.c_uint(0)) == 0
        return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_uint8)), (nbytes,))
    if kind == "new":
        return np.empty(nbytes, np.uint8)
    return np.full(nbytes + 4, 7, np.uint8)[4 if kind == "offset" else 0:][:nbytes]


# one word, rows that no group of four words divides, one band and one word
# more, eight bands, the staging's size for one plane and for two, and past it
SIZES = [(1, 1), (5, 3), (128, 256), (131, 251), (512, 256), (1027, 409), (2048, 1024), (2048, 2048), (2049, 2049),
         (3001, 2803)]


@pytest.mark.parametrize("kind", ["warm", "new", "pinned", "offset"])
@pytest.mark.parametrize("wh", SIZES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_read_back(ctx, wh, kind):
    w, h = wh
    rng = np.random.default_rng(w * h)
    color = rng.integers(0, 256, (h, w, 4), np.uint8)
    depth = rng.random((h, w), np.float32)
    t = ctx.target(w, h)
    assert ctx.lib.hana_target_upload(ctx.h, t, _u8(color), _f32(depth)) == 0
    got = [_memory(ctx, kind, 4 * w * h) for _ in range(4)]
    for _ in range(2):   # the second into what the first has touched
        assert ctx.lib.hana_target_read(ctx.h, t, _u8(got[0]), _f32(got[1])) == 0
        assert ctx.lib.hana_target_read(ctx.h, t, None, _f32(got[2])) == 0
        assert ctx.lib.hana_target_present(ctx.h, t, _u8(got[3])) == 0
        assert got[0].tobytes() == color.tobytes()
        assert got[1].tobytes() == depth.tobytes()
        assert got[2].tobytes() == depth.tobytes()
        assert got[3].tobytes() == color[::-1, :, [2, 1, 0, 3]].tobytes()
        for g in got:
            g[:] = 0
    if kind == "pinned":
        for g in got:
            assert ctx.lib.hipHostFree(C.c_void_p(g.ctypes.data)) == 0


def test_read_completes_overflowed_draw(ctx):
    """A read straight after a draw that outgrows a new context's workspace
    returns the image of the draw rendered again, not the first one's."""
    from edge_scenes import IDENTITY_VP, sliver_scene, with_camera_vp
    from hana_amd.gpu import Context, build_uniforms
    scene = sliver_scene()
    with Context(0) as c:
        u = with_camera_vp(build_uniforms(scene), IDENTITY_VP)
        args = (c.mesh(scene.mesh), scene.shader, u, c.target(scene.width, scene.height), c.texture(scene.diffuse),
                c.texture(scene.normal))
        shots = []
        for _ in range(2):
            c.clear(args[3])
            c.draw(*args)
            shots.append(c.present(args[3], scene.width, scene.height))
        assert c.replay_count() == 1
        assert np.array_equal(shots[0], shots[1])
        assert len(np.unique(shots[0])) > 16
