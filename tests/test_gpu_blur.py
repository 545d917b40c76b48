"""The recursive AO blur (Buffer1f::TwoPassGaussianBlurDenoised) against a
loop in its order, bit for bit, where its chunks of 32 samples and groups of
64 lines can go wrong: lines shorter than its 4 samples of reach, chunk
remainders, one line more than a group, rows that are not whole 16-byte
quads, an output that does not start at 16 bytes."""
import ctypes as C

import numpy as np
import pytest

import forkerrenderer_amd as F
from forkerrenderer_amd import nao as NA
from tests.test_zz_no_alloc import DevBuf, _hip
from tests.util import assert_bitexact

pytestmark = pytest.mark.gpu

W5 = np.array([0.227027, 0.1945946, 0.1216216, 0.054054, 0.016216], np.float32)


def _lines(a):
    """Blurs each row of a (lines, n) in place, sample after sample."""
    n = a.shape[1]
    for x in range(n):
        q = a[:, x] * W5[0]
        for i in range(1, 5):
            q = q + a[:, min(x + i, n - 1)] * W5[i]
            q = q + a[:, max(x - i, 0)] * W5[i]
        a[:, x] = q


@pytest.mark.parametrize("w,h,offset", [(1, 1, 0), (3, 2, 0), (4, 65, 0), (31, 33, 0), (32, 64, 0), (33, 129, 0), (36, 5, 0),
                                        (64, 64, 1), (100, 70, 0), (130, 35, 3)])
def test_recursive_blur(ctx, w, h, offset):
    hip = _hip()
    print(f"recursive blur {w}x{h} offset {offset}", flush=True)
    rng = np.random.default_rng(w * 1000 + h)
    n = w * h
    g = np.zeros((F.GBUF_PLANES, n), np.float32)
    nrm = rng.normal(size=(3, n))
    g[0:3] = nrm / np.linalg.norm(nrm, axis=0)
    g[3:6] = rng.uniform(-0.5, 0.5, (3, n)) * np.array([[min(1.0, w / h)], [1.0], [1.0]])
    depth, gbuf, ao = DevBuf(hip, 4 * n), DevBuf(hip, g.nbytes), DevBuf(hip, 4 * (n + offset))
    depth.put(rng.uniform(0.0, 1.0, n).astype(np.float32))
    gbuf.put(g)
    view = np.ascontiguousarray(F.make_lookat((0.0, 0.0, 3.0), (0.0, 0.0, 0.0)), np.float32)
    proj = np.ascontiguousarray(F.make_perspective(45.0, np.float32(w) / np.float32(h), 0.01, 20.0), np.float32)
    cfg = NA.ssao_cfg(n=16, sigma=2.0)
    cfg.range = 1.0
    fn = F.lib().fgl_ssao_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.c_int, C.c_int] + [C.c_void_p] * 5 + [C.POINTER(F.SsaoCfg)]
    out = []
    for blur in (0, 1):
        cfg.blur = blur
        ctx._chk(fn(ctx._h, w, h, view.ctypes.data, proj.ctypes.data, depth.p, gbuf.p, ao.p.value + 4 * offset,
                    C.byref(cfg)), "fgl_ssao_noalloc")
        ctx.sync()
        out.append(ao.get(n + offset)[offset:].reshape(h, w))
    for b in (depth, gbuf, ao):
        b.free()
    want = out[0].copy()
    assert n < 64 or len(np.unique(want)) > 1
    _lines(want)
    _lines(want.T)
    assert_bitexact("blurred", out[1].reshape(-1), want.reshape(-1))
