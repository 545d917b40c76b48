"""Every texture wrap and filter mode on the GPU against the oracle.

The reference's textures take ForkerGL's TextureWrapping / TextureFiltering
at load time (src/forkergl.cpp:15-16, src/model.cpp:425-426): NoWrap and
Nearest unless changed first -- the modes of every reference render.  Here
the scene carries no `texture` key and is loaded with each of the 4 x 2
modes; texture coordinates are scaled to run outside [0, 1] (negative and
above 1), so the wrap rule decides most samples.  G-buffer (albedo,
roughness, metalness and the TBN-mapped normal all come from textures),
depth and shadow map bit-exact; the 8-bit image within +-1 LSB.
"""
import os

import numpy as np
import pytest

import forkerrenderer_amd as F
from forkerrenderer_amd import scenegen as G
from tests.util import assert_bitexact, gpu_frame, lsb_stats, oracle_frame

pytestmark = pytest.mark.gpu

WRAPS = {"none": F.WRAP_NONE, "repeat": F.WRAP_REPEAT, "mirror": F.WRAP_MIRROR, "clamp": F.WRAP_CLAMP}
FILTERS = {"nearest": F.FILTER_NEAREST, "linear": F.FILTER_LINEAR}


@pytest.mark.parametrize("mode", ["deferred", "forward"])
@pytest.mark.parametrize("filt", list(FILTERS))
@pytest.mark.parametrize("wrap", list(WRAPS))
def test_texture_modes(ctx, scene_dir, wrap, filt, mode):
    d = os.path.join(scene_dir, f"tex_{mode}")
    if not os.path.exists(os.path.join(d, "tiny.scene")):
        G.tiny_scene(d, seed=61, width=120, height=80, subdiv=3, tex=32, mode=mode, shadow="grid",
                     texture=None, uv_scale=3.0, pbr=(mode == "deferred"))
    sc = F.Scene(os.path.join(d, "tiny.scene"), WRAPS[wrap], FILTERS[filt])
    for i in range(sc.info.n_textures):
        t = sc.texture(i)
        assert (t["wrap"], t["filter"]) == (WRAPS[wrap], FILTERS[filt])
    print(f"texture modes: {wrap} {filt} {mode}", flush=True)
    got = gpu_frame(ctx, sc, 16)
    want = oracle_frame(sc)
    assert (want["depth"] < 3e38).sum() > 2000
    assert_bitexact("depth", got["depth"], want["depth"])
    assert_bitexact("shadow", got["shadow"], want["shadow"])
    if mode == "deferred":
        assert_bitexact("gbuf", got["gbuf"], want["gbuf"])
    mx, frac = lsb_stats(got["image"], want["image"])
    assert frac >= 0.999, (mx, frac)



@pytest.mark.parametrize("mode", ["deferred", "forward"])
@pytest.mark.parametrize("tex,other", [(1, None), (3, None), (7, (9, 6)), (33, None), (32, (32, 16))])
def test_map_sizes(ctx, scene_dir, mode, tex, other):
    """A material's maps are kept together in 4 x 4 blocks where their sizes
    agree: sizes that are no multiple of 4, a single texel, and a map of
    another size, which stays by itself."""
    d = os.path.join(scene_dir, f"mapsize_{mode}_{tex}")
    p = G.tiny_scene(d, seed=62, width=97, height=61, subdiv=3, tex=tex, mode=mode, uv_scale=3.0, pbr=(mode == "deferred"))
    if other:
        rng = np.random.default_rng(tex)
        G.write_tga(os.path.join(d, "albedo.tga"), rng.integers(0, 256, (other[1], other[0], 3), dtype=np.uint8))
    sc = F.Scene(p)
    print(f"map sizes: {mode} {tex} {other}", flush=True)
    got = gpu_frame(ctx, sc, 16)
    want = oracle_frame(sc)
    assert_bitexact("depth", got["depth"], want["depth"])
    if mode == "deferred":
        assert_bitexact("gbuf", got["gbuf"], want["gbuf"])
    mx, frac = lsb_stats(got["image"], want["image"])
    assert frac >= 0.999, (mx, frac)


@pytest.mark.parametrize("shadow", ["hard", "pcf", "pcss", "grid"])
@pytest.mark.parametrize("mode,width,height", [("deferred", 333, 201), ("forward", 333, 201), ("deferred", 65, 5),
                                               ("forward", 1, 1)])
def test_partly_covered_frames_by_filter(ctx, scene_dir, shadow, mode, width, height):
    """The kernel of each shadow filter on frames of enough blocks to be dealt
    out in runs and of fewer, with odd edges, wavefronts nothing was drawn to
    and wavefronts that are partly covered; SSAO leaves its early ones too."""
    p = G.tiny_scene(os.path.join(scene_dir, f"part_{shadow}_{mode}_{width}"), seed=63, width=width, height=height,
                     subdiv=3, tex=16, mode=mode, shadow=shadow, ssao=(mode == "deferred"))
    sc = F.Scene(p)
    print(f"partly covered: {shadow} {mode} {width}x{height}", flush=True)
    got = gpu_frame(ctx, sc, 16)
    want = oracle_frame(sc)
    assert_bitexact("depth", got["depth"], want["depth"])
    assert_bitexact("shadow", got["shadow"], want["shadow"])
    if mode == "deferred":
        assert_bitexact("gbuf", got["gbuf"], want["gbuf"])
    mx, frac = lsb_stats(got["image"], want["image"])
    assert frac >= 0.998, (mx, frac)   # SSAO taps within rounding of a threshold


@pytest.mark.parametrize("mode", ["deferred", "forward"])
@pytest.mark.parametrize("grid", [1, 3, 4, 5, 7])
def test_grid_filter_sizes(ctx, scene_dir, mode, grid):
    """The 3 x 3 and 5 x 5 grids by rows and columns, the others texel by
    texel, on a map whose edges the grid crosses."""
    p = G.tiny_scene(os.path.join(scene_dir, f"grid_{mode}_{grid}"), seed=64, width=97, height=61, subdiv=3, tex=16,
                     mode=mode, shadowmap=23, extra=f"shadowfilter grid {grid}")
    sc = F.Scene(p)
    assert sc.info.shadow.grid == grid
    got = gpu_frame(ctx, sc, 16)
    want = oracle_frame(sc)
    assert_bitexact("shadow", got["shadow"], want["shadow"])
    mx, frac = lsb_stats(got["image"], want["image"])
    assert frac >= 0.999, (mx, frac)


@pytest.mark.parametrize("shadow", ["hard", "pcf", "pcss", "grid"])
@pytest.mark.parametrize("mode,pbr", [("deferred", True), ("deferred", False), ("forward", True), ("forward", False)])
def test_dense_meshes(ctx, scene_dir, mode, pbr, shadow):
    """Frames of fewer than two pixels a face, whose resolve makes the varyings
    from the corner records, per mode, shading and shadow filter."""
    p = G.tiny_scene(os.path.join(scene_dir, f"dense_{mode}_{pbr}_{shadow}"), seed=65, width=97, height=61, subdiv=5, tex=16,
                     mode=mode, pbr=pbr, shadow=shadow)
    sc = F.Scene(p)
    print(f"dense: {mode} pbr {pbr} {shadow}", flush=True)
    got = gpu_frame(ctx, sc, 16)
    want = oracle_frame(sc)
    assert_bitexact("depth", got["depth"], want["depth"])
    if mode == "deferred":
        assert_bitexact("gbuf", got["gbuf"], want["gbuf"])
    mx, frac = lsb_stats(got["image"], want["image"])
    assert frac >= 0.999, (mx, frac)
