"""The direct rasteriser (passes from cleared targets) against the tile lists
(passes that go on from earlier depths), bit for bit, over what their rules
divide: lanes per triangle, the workgroup's LDS box, the list of large
triangles and its runs of items, NaN depths, screens of one pixel and wider than
the exact regime, several draws with equal depths.

The second rendering (one per tile size) starts with a draw that covers
nothing and a change of state, which flushes it: the rest of the pass then
continues from existing depths and takes the tile lists.  Which way each took
is read from the kernels it ran."""
import time

import numpy as np
import pytest

import forkerrenderer_amd as F

pytestmark = pytest.mark.gpu

EYE4 = np.eye(4, dtype=np.float32)


def _model(ctx, mat, pos):
    """Separate triangles, pos (n, 3, 3) in clip space."""
    n = len(pos)
    f = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    return ctx.upload_model({"pos": pos.reshape(-1, 3).astype(np.float32), "uv": np.zeros((3 * n, 2), np.float32),
                             "nrm": np.tile(np.array([[0, 0, 1]], np.float32), (3 * n, 1)), "tan": None, "vi": f, "ti": f,
                             "ni": f, "face_material": np.full(n, mat, np.int32), "support_pbr": False})


def _triangles(rng, n, size, spread=1.1):
    """n triangles of about `size` of the screen's half width, anywhere on it."""
    c = rng.uniform(-spread, spread, (n, 1, 3)) * np.array([1, 1, 0.45])
    return c + rng.uniform(-size, size, (n, 3, 3)) * np.array([1, 1, 0.05])


def _material(ctx):
    m = F.Material()
    for f in ("map_kd", "map_ks", "map_ke", "map_bump", "map_base", "map_rough", "map_metal", "map_ao", "map_pbr_ke"):
        setattr(m, f, -1)
    return ctx.upload_material(m)


def _scene(name, rng):
    """(models, W, H): each model's triangles."""
    if name == "few_mixed":        # 16 lanes a triangle, boxes below and above the LDS box, items
        return [np.concatenate([_triangles(rng, 300, s) for s in (0.01, 0.05, 0.2, 0.9)])], 333, 201
    if name == "four_lanes":
        return [_triangles(rng, 40000, 0.02)], 900, 500
    if name == "one_lane":
        return [_triangles(rng, 270000, 0.004), _triangles(rng, 5, 1.5)], 512, 300
    if name == "full_screens":     # 1,200 full screens of 300 items each: runs of 16, many searches
        full = np.array([[-3, -3, 0], [3, -3, 0], [0, 3, 0]]) + 0.0
        return [full[None] + rng.uniform(-0.4, 0.4, (1200, 3, 1)) * np.array([0, 0, 1]), _triangles(rng, 100, 0.1)], 640, 480
    if name == "ties":             # the same triangles drawn three times: the first draw's win
        t = _triangles(rng, 200, 0.3)
        return [t, _triangles(rng, 50, 0.3), t, t[::-1]], 160, 90
    if name == "one_pixel":
        return [_triangles(rng, 50, 2.0)], 1, 1
    if name == "thin":
        return [_triangles(rng, 2000, 0.3)], 5, 300
    if name == "inexact":          # wider than 8192: the general coverage sequence
        return [_triangles(rng, 400, 0.1)], 8300, 6
    if name == "nan":              # NaN and infinite depths among ordinary ones
        t = _triangles(rng, 400, 0.4)
        t[::7, 1, 2] = np.nan
        t[3::11, 2, 2] = np.inf
        return [t, _triangles(rng, 100, 0.4)], 120, 80
    if name == "nan_large":        # the same with listed triangles before and after the marks
        t = _triangles(rng, 300, 1.0)
        t[::7, 1, 2] = np.nan
        return [_triangles(rng, 60, 0.1), t, _triangles(rng, 60, 1.0)], 640, 480
    if name == "off_screen":
        return [_triangles(rng, 500, 0.3) + np.array([9.0, 0.0, 0.0])], 100, 70
    raise AssertionError(name)


@pytest.mark.parametrize("name", ["few_mixed", "four_lanes", "one_lane", "full_screens", "ties", "one_pixel", "thin",
                                  "inexact", "nan", "nan_large", "off_screen"])
@pytest.mark.parametrize("shadow", [False, True])
def test_direct_equals_lists(ctx, name, shadow):
    rng = np.random.default_rng(len(name))
    tris, W, H = _scene(name, rng)
    mat = _material(ctx)
    models = [(_model(ctx, mat, t), EYE4) for t in tris]
    _direct_against_lists(ctx, mat, models, W, H, shadow, name, tiles=(16,) if name == "full_screens" else (8, 16, 32))


def _direct_against_lists(ctx, mat, draws, W, H, shadow, name, timed=False, tiles=(16,)):
    """draws: (model, matrix) in order.  timed: returns the ms of each
    rendering's rasterisation (a second one, so that nothing is allocated)."""
    off = _model(ctx, mat, np.full((1, 3, 3), 9.0) + np.eye(3)[None])
    ctx.set_shadow(False)
    eye = np.ascontiguousarray(EYE4)
    ctx.set_matrix(F.MAT_PROJ, eye)
    ctx.set_matrix(F.MAT_VIEW, eye)
    ctx.set_matrix(F.MAT_LIGHT_SPACE, eye)
    ctx.set_viewport(0, 0, W, H, shadow=shadow)
    out, ms = [], []
    for lists in (0,) + tiles:   # 0: direct
        print(f"direct test {name} {W}x{H} shadow {shadow} lists {lists}", flush=True)
        ctx.set_tile_size(lists or 16)
        ctx.sync()
        ctx.read_timings()
        ctx.enable_timing(True)
        if shadow:
            ctx.init_shadow_buffer(W, H)
        else:
            ctx.init_targets(W, H)
        ctx.set_eye((0.0, 0.0, 1.0))
        ctx.begin_pass(F.PASS_SHADOW if shadow else F.PASS_GEOMETRY)
        if lists:
            ctx.draw_model(off, eye)
            ctx.set_eye((0.0, 0.0, 2.0))   # flushes the pass so far
        for k, at in draws:
            ctx.draw_model(k, at)
        if timed:
            ctx.end_pass()
            ctx.sync()
            ctx.read_timings()
            ctx.init_targets(W, H)
            ctx.begin_pass(F.PASS_GEOMETRY)
            if lists:
                ctx.draw_model(off, eye)
                ctx.set_eye((0.0, 0.0, 1.0))
            for k, at in draws:
                ctx.draw_model(k, at)
        ctx.end_pass()
        ctx.sync()
        kernels = ctx.read_timings()
        ctx.enable_timing(False)
        assert ("setup" in [k for k, _ in kernels]) == (lists > 0), (lists, kernels)
        ms.append(sum(t for k, t in kernels if k in ("vertex", "setup", "scan", "emit", "sort", "tile_ranges", "raster")))
        which = (F.TARGET_SHADOW_DEPTH, F.TARGET_SHADOW) if shadow else (F.TARGET_DEPTH, F.TARGET_GBUFFER)
        out.append([ctx.read(t).view(np.uint32) for t in which])
    ctx.set_tile_size(16)
    for tile, a, b, what in [(tile, a, b, what) for tile, got in zip(tiles, out[1:])
                             for a, b, what in zip(out[0], got, ("depth", "shadow value" if shadow else "G-buffer"))]:
        if name.startswith("nan"):   # a NaN's payload is not the fold's
            na, nb = np.isnan(a.view(np.float32)), np.isnan(b.view(np.float32))
            assert np.array_equal(na, nb), what
            a, b = np.where(na, 0, a), np.where(nb, 0, b)
        assert np.array_equal(a, b), f"{what}, tile {tile}: {(a != b).sum()} of {a.size} differ"
    depth = out[0][0].view(np.float32)
    assert (depth < 3e38).any() == (name != "off_screen")
    return ms


@pytest.mark.parametrize("shadow", [False, True])
def test_many_small_draws_beside_a_large_one(ctx, shadow):
    """8,200 draws of one triangle, draws of none among and after them, and
    one of 131,072: the launches are sized by what each draw holds (their
    number times the largest draw is more workgroups than a launch takes)."""
    rng = np.random.default_rng(5)
    mat = _material(ctx)
    small = _model(ctx, mat, _triangles(rng, 1, 0.02, 0.0))
    none = _model_without_faces(ctx)
    draws = []
    for k in range(8200):
        at = EYE4.copy()
        at[0, 3], at[1, 3], at[2, 3] = rng.uniform(-1, 1), rng.uniform(-1, 1), rng.uniform(-0.4, 0.4)
        draws.append((small, np.ascontiguousarray(at)))
        if k % 1000 == 3:
            draws += [(none, EYE4)] * 2
    draws.insert(4000, (_model(ctx, mat, _triangles(rng, 131072, 0.01)), EYE4))
    draws += [(none, EYE4)] * 3
    _direct_against_lists(ctx, mat, draws, 320, 200, shadow, "many draws")


@pytest.mark.parametrize("n", [2, 7, 8, 9, 10])
@pytest.mark.parametrize("shadow", [False, True])
def test_few_draws(ctx, n, shadow):
    """Around eight draws, up to which a workgroup finds its draw in the kernel's
    arguments: draws of none first, in the middle and last."""
    rng = np.random.default_rng(n)
    mat = _material(ctx)
    none = _model_without_faces(ctx)
    models = [none if k in (0, n // 2, n - 1) and n > 2 else _model(ctx, mat, _triangles(rng, 40 + 700 * (k % 3), 0.1))
              for k in range(n)]
    _direct_against_lists(ctx, mat, [(m, EYE4) for m in models], 250, 130, shadow, f"{n} draws")


def _model_without_faces(ctx):
    f = np.zeros((0, 3), np.int32)
    return ctx.upload_model({"pos": np.ones((300, 3), np.float32), "uv": np.zeros((1, 2), np.float32),
                             "nrm": np.ones((1, 3), np.float32), "tan": None, "vi": f, "ti": f, "ni": f,
                             "face_material": np.zeros(0, np.int32), "support_pbr": False})


@pytest.mark.parametrize("nan", [False, True])
def test_large_triangles_are_shared_out(ctx, nan):
    """Layers of full-screen triangles, more of them than 2^18 items of 64 x 16
    pixels; with a NaN vertex among them the pass walks them twice.  No
    wavefront is left with whole ones: the pass takes no more than a few times
    what the tile lists take (an eighth of the layers on their own wavefronts
    took 200 times as long)."""
    rng = np.random.default_rng(3)
    W, H, n = 1920, 1080, 256
    full = np.array([[[-3, -3, 0.9], [3, -3, 0.9], [0, 3, 0.9]]]) + rng.uniform(0, 0.05, (n, 1, 1)) * np.array([0, 0, 1])
    full[5, 1, 2] = np.nan if nan else 0.9
    mat = _material(ctx)
    m = _model(ctx, mat, full)
    print("layers", nan, flush=True)
    ms = _direct_against_lists(ctx, mat, [(m, EYE4)], W, H, False, "nan layers" if nan else "layers", timed=True)
    assert ms[0] < 8 * ms[1] + 1.0, ms


def test_draws_in_front_of_the_camera_are_bounded_by_their_box(ctx):
    """Host time of a pass of many draws: models of few vertices, which are
    tried one by one where the box of the model does not clear the camera
    plane, cost no more than models of many (three times as much when they
    were tried first)."""
    rng = np.random.default_rng(9)
    mat = _material(ctx)
    ctx.set_shadow(False)
    for which in (F.MAT_PROJ, F.MAT_VIEW):
        ctx.set_matrix(which, np.ascontiguousarray(EYE4))
    ctx.set_viewport(0, 0, 64, 64)
    took = []
    for faces in (85, 86):   # 255 and 258 vertices
        m = _model(ctx, mat, _triangles(rng, faces, 0.05))
        best = 1e9
        for rep in range(6):
            ctx.init_targets(64, 64)
            ctx.begin_pass(F.PASS_GEOMETRY)
            for k in range(2000):
                ctx.draw_model(m, EYE4)
            ctx.sync()
            t0 = time.perf_counter()
            ctx.end_pass()
            best = min(best, time.perf_counter() - t0)
        took.append(best)
    print("2,000 draws, seconds:", took, flush=True)
    assert took[0] < 1.5 * took[1], took


def test_passes_of_a_frame_share_their_draw_table(ctx):
    """The draw table is written when the draws change, not when a pass takes
    another number of lanes per triangle than the one before (each write waits
    for the stream): 40,000 triangles, a shadow map of 64 x 64 (one lane) and a
    view of 640 x 400 (four)."""
    rng = np.random.default_rng(11)
    mat = _material(ctx)
    a, b = (_model(ctx, mat, _triangles(rng, 20000, 0.02)) for _ in range(2))
    ctx.set_shadow(False)
    for which in (F.MAT_PROJ, F.MAT_VIEW, F.MAT_LIGHT_SPACE):
        ctx.set_matrix(which, np.ascontiguousarray(EYE4))
    ctx.set_viewport(0, 0, 640, 400)
    ctx.set_viewport(0, 0, 64, 64, shadow=True)
    writes = []
    for order in ((a, b), (a, b), (b, a), (b, a)):
        ctx.sync()
        ctx.read_timings()
        ctx.enable_timing(True)
        ctx.init_shadow_buffer(64, 64)
        ctx.init_targets(640, 400)
        for which in (F.PASS_SHADOW, F.PASS_GEOMETRY):
            ctx.begin_pass(which)
            for m in order:
                ctx.draw_model(m, EYE4)
            ctx.end_pass()
        ctx.sync()
        names = [n for n, _ in ctx.read_timings()]
        ctx.enable_timing(False)
        assert "raster_shadow" in names and "raster" in names and "setup" not in names, names
        writes.append(names.count("draw_table"))
    assert writes == [1, 0, 1, 0], writes
