"""Batched uneven views: every target of every view of a batch equals the
single-view render of that view bit for bit -- across tile sizes,
rasteriser occupancy, graph replays and a forced pair-capacity overflow."""
import numpy as np
import pytest

import forkerrenderer_amd as F
from forkerrenderer_amd import nao as NA
from forkerrenderer_amd import views as VW

pytestmark = pytest.mark.gpu

TARGETS = [F.TARGET_DEPTH, F.TARGET_GBUFFER, F.TARGET_FRAME, F.TARGET_IMAGE, F.TARGET_SHADOW,
           F.TARGET_SHADOW_DEPTH]


def bits(a):
    a = np.ascontiguousarray(a)
    return a.view(np.uint32) if a.dtype == np.float32 else a


@pytest.fixture(scope="module")
def world(ctx):
    views = VW.uneven_views(ctx, n_views=7, seed=11, subdivs=(2, 3, 4), min_px=48 * 48, max_px=320 * 240,
                            shadow_size=256, tex=64)
    # one view without shadows, one with an extra model instance
    v = views[3].desc
    views[3] = VW.View(v.width, v.height, tuple(v.eye), tuple(v.look_at),
                       list(zip(views[3].models.tolist(), views[3].mats.reshape(-1, 4, 4))),
                       [(0, (2.0, 5.0, 5.0), (3.0, 3.0, 3.0))], shadow=None)
    v = views[5]
    extra = list(zip(v.models.tolist(), v.mats.reshape(-1, 4, 4)))
    extra.append((int(v.models[1]), F.make_model_matrix((1.2, 0.2, -0.5), 30.0, 0.4)))
    d = v.desc
    views[5] = VW.View(d.width, d.height, tuple(d.eye), tuple(d.look_at), extra,
                       [(0, (2.0, 5.0, 5.0), (3.0, 3.0, 3.0))], VW.pcf_grid(5), 256)
    net = NA.NeuralAO(ctx, batch=1, crop=64, params=NA.init_params(3))
    singles = []
    for i, view in enumerate(views):
        VW.render_view(ctx, view, VW.AO_NEURAL, net)
        out = {t: ctx.read(t).copy() for t in TARGETS if view.desc.shadow_on or t not in
               (F.TARGET_SHADOW, F.TARGET_SHADOW_DEPTH)}
        out[F.TARGET_AO] = ctx.read(F.TARGET_AO).copy()
        singles.append(out)
    yield views, net, singles
    net.close()


def check(batch, views, singles, label):
    for i, ref in enumerate(singles):
        for t, want in ref.items():
            got = batch.read(i, t)
            assert np.array_equal(bits(got), bits(want)), f"{label}: view {i} target {t}"


def test_batch_equals_single_views(ctx, world):
    views, net, singles = world
    b = VW.Batch(ctx, views, VW.AO_NEURAL, net)
    b.render()
    assert b.sync() == 0
    check(b, views, singles, "eager")
    st = b.stats()
    assert st["views"] == len(views) and st["pairs_main"] > 0 and st["pairs_main"] <= st["cap_main"]
    b.close()


@pytest.mark.parametrize("tiles,occ", [((8, 8), 1), ((32, 16), 2), ((16, 32), 8)])
def test_batch_graph_replays_across_tiles(ctx, world, tiles, occ):
    views, net, singles = world
    b = VW.Batch(ctx, views, VW.AO_NEURAL, net)
    b.set_tiles(*tiles)
    b.set_occupancy(occ)
    for rep in range(3):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"tiles {tiles} occ {occ} replay {rep}")
        ctx.sync()   # eager work on the same stream between replays
    b.close()


def kernels(ctx, b):
    """Names of the kernels of one render."""
    ctx.read_timings()
    ctx.enable_timing(True)
    b.render()
    assert b.sync() == 0
    names = {n for n, _ in ctx.read_timings()}
    ctx.enable_timing(False)
    return names


@pytest.mark.parametrize("tiles,occ", [((8, 8), 1), ((32, 16), 2), ((16, 32), 8)])
def test_which_way_a_batch_rasterises(ctx, world, tiles, occ):
    """The render that counts a plan's pairs goes through the lists, replays
    through the direct rasteriser; explicit capacities keep every replay on
    the lists (tiles, occupancy and graph replays of the list path)."""
    views, net, singles = world
    b = VW.Batch(ctx, views, VW.AO_NEURAL, net)
    b.set_tiles(*tiles)
    b.set_occupancy(occ)
    assert "batch_main_sort" in kernels(ctx, b)
    check(b, views, singles, "counting")
    assert "batch_main_sort" not in kernels(ctx, b)
    check(b, views, singles, "direct")
    st = b.stats()
    b.close()
    b = VW.Batch(ctx, views, VW.AO_NEURAL, net)
    b.set_tiles(*tiles)
    b.set_occupancy(occ)
    b.set_capacity(st["pairs_shadow"] + 1, st["pairs_main"] + 1)
    for rep in range(3):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"lists, replay {rep}")
        ctx.sync()
    assert "batch_main_sort" in kernels(ctx, b)
    b.close()


def _filters(scene_dir):
    """One configuration of each deterministic shadow filter."""
    import os
    from forkerrenderer_amd import scenegen as G
    return [F.Scene(G.tiny_scene(os.path.join(scene_dir, f"batch_{k}"), shadow=k)).info.shadow
            for k in ("hard", "pcf", "pcss", "grid")]


@pytest.mark.parametrize("kinds", [(0, 1, 2, 3), (2, 2), (1, 3), (None, None), (None, 1)])
def test_batch_of_shadow_filters(ctx, scene_dir, kinds):
    """One filter over all shadowed views, several, none."""
    cfgs = _filters(scene_dir)
    base = VW.uneven_views(ctx, n_views=len(kinds), seed=29, subdivs=(3,), min_px=48 * 48, max_px=120 * 120, shadow_size=64,
                           tex=16)
    views = []
    for v, k in zip(base, kinds):
        d = v.desc
        views.append(VW.View(d.width, d.height, tuple(d.eye), tuple(d.look_at),
                             list(zip(v.models.tolist(), v.mats.reshape(-1, 4, 4))),
                             [(0, (2.0, 5.0, 5.0), (3.0, 3.0, 3.0))], None if k is None else cfgs[k], 64))
    singles = []
    for view in views:
        VW.render_view(ctx, view)
        singles.append({t: ctx.read(t).copy() for t in TARGETS
                        if view.desc.shadow_on or t not in (F.TARGET_SHADOW, F.TARGET_SHADOW_DEPTH)})
    b = VW.Batch(ctx, views)
    for rep in range(3):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"filters {kinds}, render {rep}")
    b.close()


@pytest.mark.parametrize("name", ["camera plane", "layers", "many large"])
def test_batch_of_triangle_soups(ctx, name):
    """A vertex on one view's camera plane (the whole batch stays on the
    lists), full-screen layers enough for keys to be read first, and more
    large triangles than a wavefront has lanes."""
    rng = np.random.default_rng(11)
    views = VW.uneven_views(ctx, n_views=3, seed=31, subdivs=(2,), min_px=150 * 150, max_px=320 * 240, shadow_size=128, tex=16)
    v, d = views[1], views[1].desc
    eye, at = np.array(d.eye, np.float64), np.array(d.look_at, np.float64)
    fwd = (at - eye) / np.linalg.norm(at - eye)
    right = np.cross(fwd, (0, 1, 0))
    right /= np.linalg.norm(right)
    up = np.cross(right, fwd)

    def facing(n, dist, size, spread):   # triangles across the view, in world space
        c = eye + fwd * dist.reshape(-1, 1) + (right * rng.uniform(-1, 1, (n, 1)) + up * rng.uniform(-1, 1, (n, 1))) * spread
        return np.stack([c + right * size * a + up * size * b for a, b in ((-3, -1), (3, -1), (0, 3))], 1)
    if name == "camera plane":
        tris = facing(20, rng.uniform(1, 3, 20), 0.3, 0.6)
        tris[0, 0] = eye - fwd          # the projection's w is 1 - z of the view space
    elif name == "layers":
        tris = facing(40, rng.uniform(0.5, 1.0, 40), 4.0, 0.0)
    else:
        tris = facing(80, rng.uniform(1.0, 2.5, 80), 0.6, 0.8)
    n = len(tris)
    f = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    m = ctx.upload_model({"pos": tris.reshape(-1, 3).astype(np.float32), "uv": rng.uniform(0, 1, (3 * n, 2)).astype(np.float32),
                          "nrm": np.tile(-fwd, (3 * n, 1)).astype(np.float32), "tan": None, "vi": f, "ti": f, "ni": f,
                          "face_material": np.full(n, VW.pbr_material(ctx, 5, 16), np.int32), "support_pbr": True})
    draws = list(zip(v.models.tolist(), v.mats.reshape(-1, 4, 4))) + [(m, np.eye(4, dtype=np.float32))]
    views[1] = VW.View(d.width, d.height, tuple(d.eye), tuple(d.look_at), draws, [(0, (2.0, 5.0, 5.0), (3.0, 3.0, 3.0))],
                       VW.pcf_grid(3), 128)
    singles = []
    for view in views:
        VW.render_view(ctx, view)
        singles.append({t: ctx.read(t).copy() for t in TARGETS})
    b = VW.Batch(ctx, views)
    print("batch of", name, flush=True)
    for rep in range(3):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"{name}, render {rep}")
    assert ("batch_main_sort" in kernels(ctx, b)) == (name == "camera plane")
    b.close()


def test_batch_overflow_rerenders(ctx, world):
    views, net, singles = world
    b = VW.Batch(ctx, views, VW.AO_NEURAL, net)
    b.set_capacity(200, 300)
    b.render()
    assert b.sync() >= 1
    check(b, views, singles, "after overflow")
    st = b.stats()
    assert st["cap_main"] >= st["pairs_main"] and st["cap_shadow"] >= st["pairs_shadow"]
    b.render()
    assert b.sync() == 0
    check(b, views, singles, "graph after overflow")
    b.close()


def test_batch_without_ao(ctx, world):
    views, _, _ = world
    ref = []
    for view in views[:3]:
        VW.render_view(ctx, view, VW.AO_NONE)
        ref.append({t: ctx.read(t).copy() for t in (F.TARGET_DEPTH, F.TARGET_FRAME, F.TARGET_IMAGE)})
    b = VW.Batch(ctx, views[:3], VW.AO_NONE)
    b.render()
    b.sync()
    b.render()
    b.sync()
    check(b, views[:3], ref, "no AO")
    b.close()


def test_batch_after_tables_and_ao_buffers_move(ctx, world, scene_dir):
    """Resources the batch's captured graph addresses can move after the
    batch was planned: the context's material and texture tables when new
    uploads outgrow them, the neural-AO activations when a single-frame
    inference runs on a frame larger than the whole batch.  Replays after
    each move still equal the single-view renders."""
    import os
    from forkerrenderer_amd import scenegen as G
    views, net, singles = world
    b = VW.Batch(ctx, views, VW.AO_NEURAL, net)
    b.render()
    assert b.sync() == 0
    b.render()            # the graph is captured here
    assert b.sync() == 0
    check(b, views, singles, "before")
    # many new materials and textures: both tables are reallocated
    tex = np.zeros((4, 4, 3), np.uint8)
    m = F.Material()
    for f in ("map_kd", "map_ks", "map_ke", "map_bump", "map_base", "map_rough", "map_metal", "map_ao", "map_pbr_ke"):
        setattr(m, f, -1)
    for _ in range(300):
        ctx.upload_texture(tex)
        ctx.upload_material(m)
    for rep in range(2):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"after table growth, replay {rep}")
    # a single-frame neural AO larger than the batch moves the activations
    px = b.stats()["pixels"]
    W, H = 1024, 1 + px // 1024
    p = G.tiny_scene(os.path.join(scene_dir, "batch_big_nao"), seed=3, width=W, height=H, subdiv=2, tex=16)
    ctx.render_scene(F.Scene(p))
    net.infer()
    ctx.sync()
    for rep in range(2):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"after activation move, replay {rep}")
    b.close()


@pytest.mark.parametrize("dense", [True, False])
def test_batch_of_larger_meshes(ctx, dense):
    """More triangles than get 16 lanes whatever their size: one lane, four and
    (the grounds) sixteen.  dense: fewer than two pixels a face over all views:
    replays make the varyings from the corner records, the measuring render
    from the vertices'."""
    n, most, shadow = (4, 80, 64) if dense else (6, 560, 600)
    views = VW.uneven_views(ctx, n_views=n, seed=17, subdivs=(5,), min_px=40 * 40, max_px=most * most, shadow_size=shadow, tex=32)
    singles = []
    for view in views:
        VW.render_view(ctx, view)
        singles.append({t: ctx.read(t).copy() for t in TARGETS})
    b = VW.Batch(ctx, views)
    st = b.stats()
    assert st["tris_main"] > 32768 and (st["pixels"] < 2 * st["tris_main"]) == dense
    if not dense:   # a sphere's pixels a face, in its view and in its map
        faces = st["tris_main"] // n
        assert min(v.pixels for v in views) < 2.5 * faces < max(v.pixels for v in views) and shadow ** 2 > 7.5 * faces
    for rep in range(3):
        b.render()
        assert b.sync() == 0
        check(b, views, singles, f"dense {dense}, render {rep}")
    b.close()


def test_batch_outlives_its_context():
    c = F.Context(0)
    b = VW.Batch(c, VW.uneven_views(c, n_views=2, seed=23, subdivs=(1,), min_px=256, max_px=512, shadow_size=32, tex=16))
    for _ in range(2):   # the second captures a graph
        b.render()
        assert b.sync() == 0
    c.close()
    for call in (b.render, b.sync, b.stats, lambda: b.set_tiles(8, 8), lambda: b.set_occupancy(2), lambda: b.set_capacity(0, 0),
                 lambda: b.use_graph(False), lambda: b.read(0, F.TARGET_IMAGE)):
        with pytest.raises(F.FglError, match=r"\(-1\)"):
            call()
    b.close()
