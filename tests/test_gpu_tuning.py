"""What a batch reports as its tuning is what was run: set again, it gives the
same waves per raster."""
import numpy as np
import pytest

from test_gpu_parity import soup_scene

pytestmark = pytest.mark.gpu

# target, shadow map, waves: 2 from 10,000 tiles and 4 pixels per face on, for
# each of the two rasters (shadow maps, targets)
CASES = {"small": ((320, 200), None, 4), "large": ((1600, 1600), None, 2), "both-large": ((1600, 1600), (1600, 1600), 2),
         "differ": ((1600, 1600), (320, 200), 0)}


@pytest.mark.parametrize("tune", [False, True], ids=["finalize", "autotune"])
@pytest.mark.parametrize("name", CASES)
def test_reported_waves(name, tune):
    from hana_amd.gpu import Batch, Context, build_uniforms
    (w, h), shadow, waves = CASES[name]
    scene = soup_scene(2000, w, h, 5, 60, 7)
    scene.shadow, scene.shadow_size = shadow is not None, shadow
    with Context(0) as ctx:
        u, mesh, tex = build_uniforms(scene), ctx.mesh(scene.mesh), (ctx.texture(scene.diffuse), ctx.texture(scene.normal))
        images = []
        tuning = None
        for k in range(2):
            t, sm = ctx.target(w, h), ctx.target(*shadow) if shadow else None
            batch = Batch(ctx)
            batch.add(ctx.frame_desc(mesh, scene.shader, scene.shadow, u, t, sm, *tex))
            if tuning:
                batch.set_tuning(tuning["tile_size"], tuning["raster_wgs_per_cu"], tuning["parts"], tuning["raster_waves"])
            if tune and not tuning:
                chosen = batch.autotune(reps=1)
                assert chosen == batch.tuning()
            else:
                batch.finalize(use_graph=True)
            got = batch.tuning()
            assert not tuning or all(got[f] == tuning[f] for f in got if f != "ms")
            tuning = got
            if not tune:
                assert tuning["raster_waves"] == waves
            batch.run()
            images.append(ctx.read(t, w, h))
            batch.close()
    assert images[0][1].tobytes() == images[1][1].tobytes() and np.array_equal(images[0][0], images[1][0])
