"""Lines' and points' fragment lists over special depths: NaN among the drawn
ones; NaN, both infinities, both zeros and a subnormal among the stored ones.
One draw gives what the same primitives drawn one at a time give, bit for
bit, for every comparison, with and without depth writes and stencil; and a
drawn point's effect is the comparison's."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

from scene_runner import REPO

pytestmark = pytest.mark.gpu

STORED = np.array([np.nan, np.inf, -np.inf, -0.0, 0.0, 1e-40, 0.25, -0.5], np.float32)
DRAWN = np.array([np.nan, -0.5, -0.25, -0.0, 0.0, 0.25, 0.5], np.float32)
PASSES = [lambda d, s: False, lambda d, s: True, lambda d, s: d < s, lambda d, s: d <= s, lambda d, s: d > s,
          lambda d, s: d >= s, lambda d, s: d == s, lambda d, s: d != s]


@pytest.fixture(scope="module")
def cases():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    m.lib = C.CDLL(os.path.join(REPO, "srp_amd", "libsrp_amd.so"))
    m.lib.srpFramebufferUpload.argtypes = [C.c_void_p]
    m.lib.srpDepthWrite.argtypes = [C.c_bool]
    return m


def program(cases, a):
    return a.program("sc_vsMix", [(2, cases.T_FLOAT, cases.AFFINE), (1, cases.T_FLOAT, cases.FLAT),
                                  (1, cases.T_UINT32, cases.FLAT)], "sc_fsMix")


def vertices(rng, n, z):
    v = np.zeros((n, 8), np.float32)
    v[:, :2] = rng.uniform(-0.99, 0.99, (n, 2))
    v[:, 2], v[:, 3] = z, 1
    v[:, 4:7] = rng.random((n, 3))
    v[:, 7] = np.arange(n, dtype=np.uint32).view(np.float32)
    return v


def start(cases, a, s, fb, stored):
    """A frame whose stored depths are the given ones."""
    cases.start_frame(a, fb, 1.0, 1)
    a.FramebufferDownload(fb)
    s.images[1][:] = stored
    cases.lib.srpFramebufferUpload(fb)


@pytest.mark.parametrize("kind", ["points", "lines"])
@pytest.mark.parametrize("n,w,h", [(300, 8, 1), (1100, 2, 2), (600, 17, 11)])
@pytest.mark.parametrize("op", range(8))
def test_one_draw_equals_single_draws(cases, op, n, w, h, kind):
    a = cases.api()
    a.NewContext(a.context)
    s = cases.State("test")
    rng = np.random.default_rng(100 * op + n)
    per, prim = (2, cases.PRIM_LINES) if kind == "lines" else (1, cases.PRIM_POINTS)
    z = np.repeat(rng.choice(DRAWN, n // per), per)
    vb = s.vertices(vertices(rng, n, z), 32)
    p = program(cases, a)
    a.DepthTest(True)
    a.DepthCompareOp(op)
    a.RasterPointSize(1.0)
    a.StencilFunc(cases.CMP_ALWAYS, 0, 0xFF)
    a.StencilOp(cases.ST_KEEP, cases.ST_KEEP, cases.ST_INCR)
    fb = s.framebuffer(w, h)
    stored = STORED[np.arange(w * h) % len(STORED)]
    frames = []
    for write in (True, False):
        for single in (False, True):
            cases.lib.srpDepthWrite(write)
            start(cases, a, s, fb, stored)
            for k in range(0, n, per) if single else (0,):
                a.DrawVertexBuffer(vb, fb, C.byref(p), prim, k, per if single else n)
            a.FramebufferDownload(fb)
            frames.append([x.copy() for x in s.images])
    # (the stencil test is enabled by any call, as the reference does, so it goes last)
    a.StencilTest(True)
    cases.lib.srpDepthWrite(True)
    for single in (False, True):
        start(cases, a, s, fb, stored)
        for k in range(0, n, per) if single else (0,):
            a.DrawVertexBuffer(vb, fb, C.byref(p), prim, k, per if single else n)
        a.FramebufferDownload(fb)
        frames.append([x.copy() for x in s.images])
    for one, many in zip(frames[0::2], frames[1::2]):
        for x, y in zip(one, many):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
    if op == cases.CMP_ALWAYS:
        assert np.count_nonzero(frames[0][0])
        if w > 8:   # of a few pixels, none need end with a NaN
            assert np.isnan(frames[0][1]).any()


@pytest.mark.parametrize("op", range(8))
def test_a_run_of_points_compares_as_one_after_another(cases, op):
    """Every pair of drawn depths over every stored one, a pixel each, in one
    draw."""
    a = cases.api()
    a.NewContext(a.context)
    s = cases.State("test")
    grid = [(st, x, y) for st in STORED for x in DRAWN for y in DRAWN]
    w = len(grid)
    rng = np.random.default_rng(7)
    v = vertices(rng, 2 * w, np.array([g[1] for g in grid] + [g[2] for g in grid], np.float32))
    v[:, 0] = np.tile((np.arange(w) + 0.5) / w * 2 - 1, 2)
    v[:, 1] = 0
    p = program(cases, a)
    a.DepthTest(True)
    a.DepthCompareOp(op)
    a.RasterPointSize(1.0)
    cases.lib.srpDepthWrite(True)
    fb = s.framebuffer(w, 1)
    start(cases, a, s, fb, np.array([g[0] for g in grid], np.float32))
    vb = s.vertices(v, 32)
    a.DrawVertexBuffer(vb, fb, C.byref(p), cases.PRIM_POINTS, 0, 2 * w)
    a.FramebufferDownload(fb)
    want, drawn = [], []
    for st, x, y in grid:
        hit = False
        for d in (x, y):
            if PASSES[op](d, st):
                st, hit = d, True
        want.append(st)
        drawn.append(hit)
    want = np.array(want, np.float32)
    got = s.images[1]
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))
    assert np.array_equal(s.images[0] != 0, np.array(drawn))
