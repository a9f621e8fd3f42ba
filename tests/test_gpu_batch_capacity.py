"""A batch whose vertices change on the device behind the API (which then
cannot size it again): frames with more records than its buffers hold draw the
first of them and nothing else, whatever the rest of the buffers holds, and
say so."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

from scene_runner import REPO

pytestmark = pytest.mark.gpu

SIDE, N = 256, 200
DATA_OFFSET = 24   # of SRPVertexBuffer's device pointer: after three sizes
CALLBACK = C.CFUNCTYPE(None, C.c_int, C.c_int, C.c_char_p, C.c_char_p, C.c_void_p)


class Callback(C.Structure):
    _fields_ = [("fn", CALLBACK), ("userParameter", C.c_void_p)]


@pytest.fixture(scope="module")
def cases():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    m.lib = C.CDLL(os.path.join(REPO, "srp_amd", "libsrp_amd.so"))
    m.lib.srpSetMessageCallback.argtypes = [Callback]
    m.lib.srpBatchInfo.argtypes = [C.c_void_p, C.c_void_p]
    m.lib.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    return m


def triangles(size, hidden):
    """N triangles with boxes of `size` pixels; the first `hidden` are moved
    out of the view."""
    rng = np.random.default_rng(int(size))
    p = rng.uniform(0.5, SIDE - 0.5 - size, (N, 1, 2)) + size * np.array([[0.0, 0.1], [1.0, 0.0], [0.3, 1.0]])
    p[:hidden, :, 0] -= 2 * SIDE
    v = np.concatenate([p / (SIDE / 2) - 1, rng.uniform(-0.9, 0.9, (N, 3, 1)), rng.random((N, 3, 3))], -1)
    return np.ascontiguousarray(v.reshape(-1, 6), np.float32)


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("size", [7.0, 40.0])
def test_records_beyond_the_capacity_are_dropped(cases, size, captured):
    a = cases.api()
    a.NewContext(a.context)
    a.DepthTest(True)
    a.DepthCompareOp(cases.CMP_LESS)
    s = cases.State("test")
    shown = N // 2
    first, now = triangles(250.0, N - shown), triangles(size, 0)
    vb = s.vertices(first, 24)
    p = a.program("sc_vsColorPass", [(3, cases.T_FLOAT, cases.PERSPECTIVE)], "sc_fsColor")
    fb = s.framebuffer(SIDE, SIDE)
    cmd = (cases.DrawCommand * 1)(cases.DrawCommand(None, vb, fb, C.pointer(p), cases.PRIM_TRIANGLES, 0, 3 * N,
                                                   C.addressof(a.context), 1, 1.0, 0))
    batch = s.own("FreeBatch", a.NewBatch(cmd, 1))
    info = (C.c_uint64 * 4)()
    cases.lib.srpBatchInfo(batch, info)
    assert info[1] == shown
    capacity = (shown + 64) * 9 // 8   # batchSize: 64 more, and an eighth
    assert shown < capacity < N
    if captured:
        assert a.BatchCapture(batch) == 0
    a.BatchRender(batch)
    a.FramebufferDownload(fb)
    address = C.c_void_p.from_address(vb + DATA_OFFSET).value
    assert cases.lib.hipMemcpy(address, now.ctypes.data, now.nbytes, 1) == 0
    said = []

    @CALLBACK
    def listen(kind, severity, function, text, user):
        said.append((function, text))

    frames = []
    cases.lib.srpSetMessageCallback(Callback(listen, None))
    try:
        for _ in range(3):
            a.BatchRender(batch)
            a.FramebufferDownload(fb)
            frames.append([x.copy() for x in s.images])
        cases.lib.srpBatchInfo(batch, info)
    finally:
        cases.lib.srpSetMessageCallback(Callback(CALLBACK(), None))
    assert any(fn == b"srpBatchRender" and b"exceeded" in text for fn, text in said), said
    cases.start_frame(a, fb)
    a.DrawVertexBuffer(s.vertices(now, 24), fb, C.byref(p), cases.PRIM_TRIANGLES, 0, 3 * capacity)
    a.FramebufferDownload(fb)
    assert np.count_nonzero(s.images[0])
    for got in frames:
        for x, y in zip(got, s.images):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
