"""A framebuffer's arrays on their way to the device and back: sizes whose
arrays end inside a sixteen-byte line, and host arrays that a caller put in
place of the framebuffer's own."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

from scene_runner import REPO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (16, 1), (67, 61), (641, 359), (1536, 1030)])
def test_arrays_survive_the_round_trip(w, h, own):
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    cases = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(cases)
    a = cases.api()
    fb = a.NewFramebuffer(w, h)
    f = cases.Framebuffer.from_address(fb)
    rng = np.random.default_rng(w)
    n = w * h
    kinds = (("color", C.c_uint32), ("depth", C.c_float), ("stencil", C.c_uint8))
    fields = {k: getattr(f, k) for k, _ in kinds}
    address = dict(fields)
    mine = {k: np.zeros(n * C.sizeof(t) + 16, np.uint8) for k, t in kinds}
    if not own:
        for k, _ in kinds:
            setattr(f, k, mine[k].ctypes.data)
            address[k] = mine[k].ctypes.data
    views = {k: np.frombuffer((C.c_uint8 * (n * C.sizeof(t))).from_address(address[k]), np.uint8) for k, t in kinds}
    want = {}
    lib = C.CDLL(os.path.join(REPO, "srp_amd", "libsrp_amd.so"))
    lib.srpFramebufferUpload.argtypes = [C.c_void_p]
    a.FramebufferSetDeferred(fb, True)
    a.FramebufferDownload(fb)
    for k, _ in kinds:
        views[k][:] = want[k] = rng.integers(0, 256, views[k].size, dtype=np.uint8)
    lib.srpFramebufferUpload(fb)
    for k, _ in kinds:
        views[k][:] = 0
    a.FramebufferDownload(fb)
    got = {k: views[k].copy() for k, _ in kinds}
    for k, _ in kinds:
        assert not mine[k][views[k].size:].any()
        setattr(f, k, fields[k])
    a.FreeFramebuffer(fb)
    for k, _ in kinds:
        assert np.array_equal(got[k], want[k]), k
