"""The autotuners try the settings that a scene's or a batch's renders use, and
no others: passes through the tile lists have tiles, the direct rasteriser's
have none."""
import os

import numpy as np
import pytest

import forkerrenderer_amd as F
from forkerrenderer_amd import autotune as A
from forkerrenderer_amd import scenegen as G
from forkerrenderer_amd import views as VW

pytestmark = pytest.mark.gpu


@pytest.fixture
def tiles(ctx):
    was = ctx.pass_tile_size(F.PASS_SHADOW), ctx.pass_tile_size(F.PASS_GEOMETRY)
    yield
    ctx.set_pass_tile_size(F.PASS_SHADOW, was[0])
    ctx.set_pass_tile_size(F.PASS_GEOMETRY, was[1])


@pytest.mark.parametrize("mode,extra,listed", [("deferred", "", set()), ("forward", "", set()),
                                               ("forward", "shadowfilter refpcf", {"main"})])
def test_scene(ctx, scene_dir, tiles, mode, extra, listed):
    p = G.tiny_scene(os.path.join(scene_dir, f"tune_{mode}_{len(extra)}"), seed=70, width=97, height=61, subdiv=3, tex=16,
                     mode=mode, extra=extra)
    sc = F.Scene(p)
    ctx.set_pass_tile_size(F.PASS_SHADOW, 32)
    ctx.set_pass_tile_size(F.PASS_GEOMETRY, 8)
    ctx.render_scene(sc)
    assert A.listed_passes(ctx, sc) == listed
    best, table = A.autotune(ctx, sc, reps=1)
    mains = (8, 16, 32) if "main" in listed else (8,)
    assert set(table) == {f"32/{t}" for t in mains}
    assert best["shadow"] == 32 and best["main"] in mains
    assert (ctx.pass_tile_size(F.PASS_SHADOW), ctx.pass_tile_size(F.PASS_GEOMETRY)) == (32, best["main"])


def _views(ctx, bad_depth):
    """Two views; bad_depth: one has a vertex on its camera plane."""
    views = VW.uneven_views(ctx, n_views=2, seed=19, subdivs=(2,), min_px=48 * 48, max_px=64 * 64, shadow_size=64, tex=16)
    if bad_depth:
        m = VW.sphere_model(1, 3, 0)
        eye, at = np.array(views[0].desc.eye, np.float64), np.array(views[0].desc.look_at, np.float64)
        m["pos"][0] = eye + (eye - at) / np.linalg.norm(eye - at)   # the projection's w is 1 - z of the view space
        m["face_material"][:] = VW.pbr_material(ctx, 3, 16)
        d = views[0].desc
        draws = list(zip(views[0].models.tolist(), views[0].mats.reshape(-1, 4, 4))) + [(ctx.upload_model(m), np.eye(4))]
        views[0] = VW.View(d.width, d.height, tuple(d.eye), tuple(d.look_at), draws, [(0, (2.0, 5.0, 5.0), (3.0, 3.0, 3.0))],
                           VW.pcf_grid(3), 64)
    return views


@pytest.mark.parametrize("bad_depth", [False, True])
def test_batch(ctx, bad_depth):
    b = VW.Batch(ctx, _views(ctx, bad_depth))
    b.set_tiles(32, 8)
    b.set_occupancy(2)
    best, table = A.autotune_batch(b, tiles=(8, 32), occupancies=(2, 4), margins=(1.0,), reps=1)
    if bad_depth:
        assert len(table) == 9 and (best["shadow_tile"], best["main_tile"]) == b.tiles
    else:
        assert set(table) == {"32/8/2/auto"} and b.tiles == (32, 8) and b.occupancy == 2
    b.close()
