"""Lines' and points' fragment lists: many primitives on few pixels in one
draw give what the same primitives drawn one at a time give, bit for bit,
for every depth comparison, with and without depth writes, scissor and
stencil, with runs of one pixel inside, across and over many of a block's
256 fragments."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

from scene_runner import REPO

pytestmark = pytest.mark.gpu

LIB = os.path.join(REPO, "srp_amd", "libsrp_amd.so")


@pytest.fixture(scope="module")
def cases():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def vertices(rng, n):
    """clip, st, level, tag of the mix shaders, depths from few values."""
    v = np.zeros((n, 8), np.float32)
    v[:, :2] = rng.uniform(-0.99, 0.99, (n, 2))
    v[:, 2] = rng.choice(np.array([-0.5, -0.25, -0.0, 0.0, 0.25, 0.5], np.float32), n) + \
        rng.choice(np.array([0, 0, 1e-3], np.float32), n)
    v[:, 3] = 1
    v[:, 4:7] = rng.random((n, 3))
    v[:, 7] = np.arange(n, dtype=np.uint32).view(np.float32)
    return v


@pytest.mark.parametrize("kind", ["points", "lines"])
@pytest.mark.parametrize("n,w,h", [(3, 2, 1), (700, 2, 1), (600, 17, 11)])
@pytest.mark.parametrize("op", range(8))
def test_one_draw_equals_single_draws(cases, op, n, w, h, kind):
    a = cases.api()
    a.NewContext(a.context)
    s = cases.State("test")
    rng = np.random.default_rng(op)
    per = 2 if kind == "lines" else 1
    prim = cases.PRIM_LINES if kind == "lines" else cases.PRIM_POINTS
    data = vertices(rng, n)
    vb = s.vertices(data, 32)
    p = a.program("sc_vsMix", [(2, cases.T_FLOAT, cases.AFFINE), (1, cases.T_FLOAT, cases.FLAT),
                               (1, cases.T_UINT32, cases.FLAT)], "sc_fsMix")
    n -= n % per
    frames = []
    for single in (False, True):
        fb = s.framebuffer(w, h)
        a.DepthTest(True)
        a.DepthCompareOp(op)
        a.RasterPointSize(1.0)
        for setup in range(5):
            C.CDLL(LIB).srpDepthWrite(C.c_bool(setup != 4))
            a.ScissorTest(setup == 1)
            a.ScissorOptions(1, 0, max(w - 3, 1), h)
            a.StencilTest(setup in (2, 3))
            a.StencilFunc(cases.CMP_ALWAYS if setup == 2 else cases.CMP_LESS, 3, 0x0F)
            a.StencilOp(0 if setup == 2 else cases.ST_INCR, cases.ST_INCR, cases.ST_INCR)
            cases.start_frame(a, fb, 0.125, 1)
            if single:
                for k in range(0, n, per):
                    a.DrawVertexBuffer(vb, fb, C.byref(p), prim, k, per)
            else:
                a.DrawVertexBuffer(vb, fb, C.byref(p), prim, 0, n)
            a.FramebufferDownload(fb)
            frames.append([x.copy() for x in s.images])
    for one, many in zip(frames[:5], frames[5:]):
        for x, y in zip(one, many):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


@pytest.mark.parametrize("order", ["sorted", "mixed"])
def test_line_draws_equal_the_edges_of_flat_triangles(cases, order):
    """Lines of 0 to 40 samples and of some hundreds and thousands, in every
    place of a wave, against the same lines walked by one lane each: the
    three edges of triangles whose last two corners are one point."""
    a = cases.api()
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LEQUAL)
    s = cases.State("test")
    w, h = 2048, 32
    rng = np.random.default_rng(5)
    length = np.concatenate([np.arange(0, 41), [63, 64, 255, 256, 257, 700, 2000, 2047], rng.integers(0, 60, 120)])
    if order == "mixed":
        length = rng.permutation(length)
    n = len(length)
    v = np.zeros((n, 2, 8), np.float32)
    start = rng.uniform(0, np.maximum(w - 1 - length, 1))
    v[:, 0, 0], v[:, 1, 0] = start / w * 2 - 1, (start + length) / w * 2 - 1
    v[:, :, 1] = rng.uniform(-0.99, 0.99, (n, 2))
    v[:, :, 2] = rng.uniform(-0.5, 0.5, (n, 2))
    v[:, :, 3] = 1
    v[:, :, 4:6] = rng.random((n, 2, 2))
    v[:, :, 6] = rng.random((n, 1))
    edges = v[:, [0, 1, 1, 1, 1, 0]].reshape(-1, 8)
    corners = v[:, [0, 1, 1]].reshape(-1, 8)
    p = a.program("sc_vsMix", [(2, cases.T_FLOAT, cases.AFFINE), (1, cases.T_FLOAT, cases.FLAT),
                               (1, cases.T_UINT32, cases.FLAT)], "sc_fsMix")
    fb = s.framebuffer(w, h)
    frames = []
    for data, prim in ((edges, cases.PRIM_LINES), (corners, cases.PRIM_TRIANGLES)):
        vb = s.vertices(np.ascontiguousarray(data, np.float32), 32)
        a.RasterPolygonMode(cases.MODES["line"] if prim == cases.PRIM_TRIANGLES else cases.MODES["fill"])
        cases.start_frame(a, fb)
        a.DrawVertexBuffer(vb, fb, C.byref(p), prim, 0, len(data))
        a.FramebufferDownload(fb)
        frames.append([x.copy() for x in s.images])
    assert np.count_nonzero(frames[0][0]) > 4000
    for x, y in zip(*frames):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
