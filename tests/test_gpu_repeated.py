"""One small draw issued again and again while the contents of its vertex
buffer change in place: counts that stay, shrink and grow, triangles that turn
from masked ones into spans, lists that outgrow the buffers sized from the
draw's last counts, and triangles that start to be clipped.  Every frame
equals the same triangles drawn for the first time, from a buffer of their
own."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

from scene_runner import REPO

pytestmark = pytest.mark.gpu

SIDE = 256


@pytest.fixture(scope="module")
def cases():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def triangles(kind, n):
    """n triangles with boxes of `size` pixels inside the view; of "half",
    every second lies outside it (no records); of "clipped", every fifth
    reaches over its left edge."""
    rng = np.random.default_rng(n)
    size = {"spans": 40.0, "view": 254.0}.get(kind, 7.0)
    corner = rng.uniform(0.5, SIDE - 0.5 - size, (n, 1, 2))
    p = corner + size * np.array([[0.0, 0.1], [1.0, 0.0], [0.3, 1.0]])
    if kind == "half":
        p[1::2, :, 0] -= 2 * SIDE
    if kind == "clipped":
        p[::5, 0, 0] = -20
    v = np.concatenate([p / (SIDE / 2) - 1, rng.uniform(-0.9, 0.9, (n, 3, 1)), rng.random((n, 3, 3))], -1)
    return np.ascontiguousarray(v.reshape(-1, 6), np.float32)


# the unclipped draws that follow "small" outgrow its spans (none), then "spans" its pairs, "half" its records
SEQUENCE = ["small", "small", "half", "small", "spans", "view", "view", "spans", "small", "clipped", "clipped", "small",
            "small", "view", "half", "small"]


@pytest.mark.parametrize("deferred", [True, False])
@pytest.mark.parametrize("n", [16, 17, 4096])
def test_contents_change_between_repeated_draws(cases, n, deferred):
    a = cases.api()
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LESS)
    s = cases.State("test")
    p = a.program("sc_vsColorPass", [(3, cases.T_FLOAT, cases.PERSPECTIVE)], "sc_fsColor")
    fb = s.framebuffer(SIDE, SIDE, deferred)

    def frame(vb):
        cases.start_frame(a, fb)
        a.DrawVertexBuffer(vb, fb, C.byref(p), cases.PRIM_TRIANGLES, 0, 3 * n)
        if deferred:
            a.FramebufferDownload(fb)
        return [x.copy() for x in s.images]

    data = {kind: triangles(kind, n) for kind in SEQUENCE}
    first = {kind: frame(s.vertices(v, 24)) for kind, v in data.items()}
    vb = s.vertices(data["small"], 24)
    for turn, kind in enumerate(SEQUENCE):
        a.VertexBufferCopyData(vb, 24, data[kind].nbytes, data[kind].ctypes.data)
        got = frame(vb)
        assert np.count_nonzero(got[0]), (turn, kind)
        for x, y in zip(first[kind], got):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (turn, kind)
