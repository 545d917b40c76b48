"""Device memory that the faster paths can do without: with no room for it the
calls still succeed, through the separate maps and the tile lists, and their
results are those with room.  The rest of the card's memory is held by the
test while a call runs, all but what the call needs without it."""
import ctypes as C

import numpy as np
import pytest

import forkerrenderer_amd as F
from forkerrenderer_amd import views as VW
from tests.test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu

MB = 1 << 20
EYE4 = np.eye(4, dtype=np.float32)


class Held:
    """Every byte of device memory but about `left`."""

    def __init__(self, left):
        self.hip, self.blocks = _hip(), []
        small = []
        for size in (4096 * MB, 256 * MB, 16 * MB):
            while True:
                p = C.c_void_p()
                if self.hip.hipMalloc(C.byref(p), size) != 0:
                    self.hip.hipGetLastError()
                    break
                (small if size == 16 * MB else self.blocks).append(p)
        # given back from 16 MiB blocks, and a larger one where those are few
        while len(small) * 16 * MB < left:
            self.hip.hipFree(self.blocks.pop())
            for _ in range(256 * MB // (16 * MB)):
                p = C.c_void_p()
                if self.hip.hipMalloc(C.byref(p), 16 * MB) == 0:
                    small.append(p)
                else:
                    self.hip.hipGetLastError()
        for _ in range(-(-left // (16 * MB))):
            self.hip.hipFree(small.pop())
        self.blocks += small

    def __enter__(self):
        return self

    def __exit__(self, *a):
        for p in self.blocks:
            self.hip.hipFree(p)
        self.blocks = []


def _free(hip):
    a, b = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def _world(ctx, tex):
    mat = VW.pbr_material(ctx, 7, tex)
    return mat, VW.upload_ground(ctx, mat), VW.upload_sphere(ctx, 3, 7, mat)


def _draws(ground, sphere):
    return [(ground, F.make_model_matrix((0.0, -1.1, 0.0), 0.0, 3.0)),
            (sphere, F.make_model_matrix((0.0, 0.0, 0.0), 30.0, 1.0))]


def _geometry(ctx, draws, W, H, started=lambda: None):
    view = np.ascontiguousarray(F.make_lookat((0.3, 1.5, 3.2), (0.0, -0.2, 0.0)), np.float32)
    proj = np.ascontiguousarray(F.make_perspective(45.0, np.float32(W) / np.float32(H), 0.01, 20.0), np.float32)
    ctx.set_shadow(False)
    ctx.set_matrix(F.MAT_VIEW, view)
    ctx.set_matrix(F.MAT_PROJ, proj)
    ctx.set_viewport(0, 0, W, H)
    ctx.init_targets(W, H)
    held = started()
    try:
        ctx.begin_pass(F.PASS_GEOMETRY)
        for m, at in draws:
            ctx.draw_model(m, at)
        ctx.end_pass()
        ctx.sync()
    finally:
        if held:
            held.__exit__()
    return ctx.read(F.TARGET_DEPTH).view(np.uint32), ctx.read(F.TARGET_GBUFFER).view(np.uint32)


def test_pass_without_room_for_keys():
    """The key plane of 4096 x 4096 pixels is 128 MiB, the lists' winners 64."""
    W = H = 4096
    with_room, without = F.Context(0), F.Context(0)
    try:
        out = []
        for c, left in ((with_room, None), (without, 112 * MB)):
            _, ground, sphere = _world(c, 64)
            _geometry(c, _draws(ground, sphere), 64, 64)   # kernels loaded, small buffers there
            print("pass with", "all memory" if left is None else f"{left // MB} MiB left", flush=True)
            out.append(_geometry(c, _draws(ground, sphere), W, H, (lambda: Held(left)) if left else (lambda: None)))
        for a, b in zip(*out):
            assert np.array_equal(a, b)
    finally:
        with_room.close()
        without.close()


def test_upload_without_room_for_bundles():
    """A 4096 x 4096 bundle is 128 MiB; the maps by themselves do as well."""
    c = F.Context(0)
    try:
        mat = VW.pbr_material(c, 9, 4096)
        print("upload with 48 MiB left", flush=True)
        with Held(48 * MB):
            alone = VW.upload_sphere(c, 3, 7, mat)
            ground = VW.upload_ground(c, mat)
        a = _geometry(c, _draws(ground, alone), 333, 201)
        bundled = VW.upload_sphere(c, 3, 7, mat)   # there is room for the bundle now
        b = _geometry(c, _draws(ground, bundled), 333, 201)
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
    finally:
        c.close()


def test_batch_without_room_for_keys():
    """A batch planned with room for all but its key plane renders through the
    lists, in every replay."""
    hip = _hip()
    c = F.Context(0)
    try:
        _, ground, sphere = _world(c, 64)
        view = VW.View(4096, 3072, (0.3, 1.5, 3.2), (0.0, -0.2, 0.0), _draws(ground, sphere),
                       [(0, (2.0, 5.0, 5.0), (3.0, 3.0, 3.0))], VW.pcf_grid(3), 1024)

        def render(b):
            out = []
            for _ in range(3):
                b.render()
                assert b.sync() == 0
                out.append([b.read(0, t) for t in (F.TARGET_DEPTH, F.TARGET_IMAGE, F.TARGET_SHADOW)])
            b.close()
            for later in out[1:]:
                assert all(np.array_equal(x, y) for x, y in zip(out[0], later))
            return out[0]

        c.sync()
        before = _free(hip)
        b = VW.Batch(c, [view])
        took = before - _free(hip)
        want = render(b)
        print(f"batch of {took // MB} MiB with {(took - 48 * MB) // MB} MiB left", flush=True)
        with Held(took - 48 * MB):
            b = VW.Batch(c, [view])
        got = render(b)
        assert all(np.array_equal(x, y) for x, y in zip(want, got))
    finally:
        c.close()
