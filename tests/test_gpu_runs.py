"""The batched rasteriser's pixel-parallel runs on lists that alternate
between triangles with and without exact masks, and with varyings below, at
and above the words a run stages: every frame equals the one-lane-per-pixel
rasteriser's, bit for bit."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

from scene_runner import REPO

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cases():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def triangles(n, size, seed):
    """n clip-space triangles, every third small (masked when binned), the
    others `size` wide, in random depth order; the first spans the view."""
    rng = np.random.default_rng(seed)
    half = np.where(np.arange(n) % 3 == 2, 0.03, size)[:, None, None]
    xy = rng.uniform(-1, 1, (n, 1, 2)) + half * rng.uniform(-1, 1, (n, 3, 2))
    xy[0] = [[-0.8, -0.8], [0.8, -0.7], [0.1, 0.9]]
    v = np.concatenate([xy, rng.uniform(-0.9, 0.9, (n, 3, 1)), rng.random((n, 3, 3))], -1)
    return np.ascontiguousarray(v.reshape(-1, 6), np.float32)


@pytest.mark.parametrize("words", [3, 8, 9, 12])
@pytest.mark.parametrize("n,size,w,h", [(1, 0.9, 40, 24), (9, 0.5, 64, 64), (400, 0.25, 333, 211)])
def test_mixed_lists_equal_the_lane_per_pixel_rasteriser(cases, words, n, size, w, h):
    a = cases.api()
    lib = C.CDLL(os.path.join(REPO, "srp_amd", "libsrp_amd.so"))
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LESS)
    s = cases.State("test")
    v = triangles(n, size, 11 * n + words)
    vb = s.vertices(v, 24)
    # the shader writes three words; the others are declared and never read
    extra = [(words - 3, cases.T_FLOAT, cases.FLAT)] if words > 3 else []
    p = a.program("sc_vsColorPass", [(3, cases.T_FLOAT, cases.PERSPECTIVE)] + extra, "sc_fsColor")
    fb = s.framebuffer(w, h)
    frames = []
    try:
        for batched in (0, 1):
            lib.srpHipSetRasterOptions(batched, 1, 24)
            cases.start_frame(a, fb)
            a.DrawVertexBuffer(vb, fb, C.byref(p), cases.PRIM_TRIANGLES, 0, 3 * n)
            a.FramebufferDownload(fb)
            frames.append([x.copy() for x in s.images])
    finally:
        lib.srpHipSetRasterOptions(1, 1, 24)
    assert np.count_nonzero(frames[0][0])
    for x, y in zip(*frames):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


def boxes(n, seed):
    """n triangles with boxes from one pixel to just above the largest that
    is masked, at every alignment to the 8x8 tiles of a 256x256 frame."""
    rng = np.random.default_rng(seed)
    k = np.arange(n)
    x0, y0 = (k * 5) % 229 + 0.25, (k * 3) % 231 + 0.25
    bw, bh = k % 26 + 0.4, (k // 26) % 26 + 0.4
    px = np.stack([x0, x0 + bw, x0 + bw * rng.random(n)], -1)
    py = np.stack([y0 + bh * rng.random(n), y0, y0 + bh], -1)
    v = np.concatenate([(px / 128 - 1)[..., None], (1 - py / 128)[..., None], rng.uniform(-0.9, 0.9, (n, 3, 1)), rng.random((n, 3, 3))], -1)
    return np.ascontiguousarray(v.reshape(-1, 6), np.float32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 676, 65535, 65536, 65537])
def test_lanes_per_triangle_do_not_change_the_frame(cases, n):
    """The first draw of n triangles and the last n of a draw of more than
    the limit of the row-parallel assembly give the same frame (the first
    triangles of the larger draw lie outside the view)."""
    a = cases.api()
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LESS)
    s = cases.State("test")
    v = boxes(n, n)
    pad = max(0, 65600 - n)
    far = np.tile(np.array([5, 5, 0, 0, 0, 0], np.float32), (3 * pad, 1))
    p = a.program("sc_vsColorPass", [(3, cases.T_FLOAT, cases.PERSPECTIVE)], "sc_fsColor")
    frames = []
    for data in (v, np.ascontiguousarray(np.concatenate([far, v]))):
        vb = s.vertices(data, 24)
        fb = s.framebuffer(256, 256)
        cases.start_frame(a, fb)
        a.DrawVertexBuffer(vb, fb, C.byref(p), cases.PRIM_TRIANGLES, 0, len(data))
        a.FramebufferDownload(fb)
        frames.append([x.copy() for x in s.images])
    for x, y in zip(*frames):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1023, 1024, 1025, 4096, 4097])
def test_repeated_small_draws_do_not_change_the_frame(cases, n):
    """A draw seen before is enqueued whole, its emitting blocks adding up
    the counts before theirs: the same frame as the first time, also after
    the vertices moved (other counts, same number) and back."""
    a = cases.api()
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LESS)
    s = cases.State("test")
    v = boxes(n, n)
    moved = v.copy()
    moved[:, 0] += np.float32(0.37)
    p = a.program("sc_vsColorPass", [(3, cases.T_FLOAT, cases.PERSPECTIVE)], "sc_fsColor")
    frames = {}
    for name, data in (("v", v), ("m", moved)):
        vb = s.vertices(data, 24)
        fb = s.framebuffer(256, 256)
        for turn in range(3):
            cases.start_frame(a, fb)
            a.DrawVertexBuffer(vb, fb, C.byref(p), cases.PRIM_TRIANGLES, 0, len(data))
            a.FramebufferDownload(fb)
            got = [x.copy() for x in s.images]
            for x, y in zip(frames.setdefault(name, got), got):
                assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


@pytest.mark.parametrize("w,h", [(16, 8), (40, 128), (24, 136), (64, 1032)])
def test_clipped_spans_in_one_draw_equal_single_draws(cases, w, h):
    """Triangles that reach over the view on every side: fans of several
    spans each, over fewer tile rows than a group has lanes, as many, one
    more, and many times as many."""
    a = cases.api()
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LESS)
    s = cases.State("test")
    n = 60
    rng = np.random.default_rng(h)
    v = np.concatenate([rng.uniform(-5, 5, (n, 3, 2)), rng.uniform(-1.5, 1.5, (n, 3, 1)), rng.random((n, 3, 3))], -1)
    v[0, :, :3] = [[-4, -4, 0.9], [4, -4, 0.9], [0, 5, 0.9]]   # covers the view
    vb = s.vertices(np.ascontiguousarray(v.reshape(-1, 6), np.float32), 24)
    p = a.program("sc_vsColorPass", [(3, cases.T_FLOAT, cases.PERSPECTIVE)], "sc_fsColor")
    fb = s.framebuffer(w, h)
    frames = []
    for calls in ([(0, 3 * n)], [(3 * k, 3) for k in range(n)]):
        cases.start_frame(a, fb)
        for first, count in calls:
            a.DrawVertexBuffer(vb, fb, C.byref(p), cases.PRIM_TRIANGLES, first, count)
        a.FramebufferDownload(fb)
        frames.append([x.copy() for x in s.images])
    assert np.count_nonzero(frames[0][0]) > w * h // 2
    for x, y in zip(*frames):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
