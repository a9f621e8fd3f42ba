"""A framebuffer's host arrays belong to the caller again when a library call
that reads them returns, however busy the device is, and whatever a clear or
the program then writes there."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest
import torch

from scene_runner import REPO

pytestmark = pytest.mark.gpu

KINDS = (("color", 4), ("depth", 4), ("stencil", 1))


@pytest.fixture(scope="module")
def api():
    spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(REPO, "perf", "cases.py"))
    cases = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(cases)
    a = cases.api()
    a.lib = C.CDLL(os.path.join(REPO, "srp_amd", "libsrp_amd.so"))
    a.lib.srpHipGetStream.restype = C.c_void_p
    a.Fields = cases.Framebuffer
    return a


def bytes_at(address, n):
    return np.frombuffer((C.c_uint8 * n).from_address(address), np.uint8)


def host_arrays(a, fb):
    f = a.Fields.from_address(fb)
    return {k: bytes_at(getattr(f, k), f.size * n) for k, n in KINDS}


def keep_busy(a):
    """Some twenty milliseconds of work on the library's stream."""
    x = torch.zeros(1 << 27, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.ExternalStream(a.lib.srpHipGetStream())):
        for _ in range(100):
            x.add_(1.0)
    return x


@pytest.mark.parametrize("own", [True, False])
def test_switch_to_deferred_takes_the_arrays_as_they_are(api, own):
    w, h = 641, 359
    fb = api.NewFramebuffer(w, h)
    f = api.Fields.from_address(fb)
    fields = {k: getattr(f, k) for k, _ in KINDS}
    mine = {k: np.zeros(w * h * n, np.uint8) for k, n in KINDS}
    if not own:
        for k, _ in KINDS:
            setattr(f, k, mine[k].ctypes.data)
    views = host_arrays(api, fb)
    rng = np.random.default_rng(1)
    want = {}
    for k, v in views.items():
        v[:] = want[k] = rng.integers(0, 256, v.size, dtype=np.uint8)
    busy = keep_busy(api)
    api.FramebufferSetDeferred(fb, True)
    for v in views.values():
        v[:] = 0
    api.FramebufferDownload(fb)
    got = {k: v.copy() for k, v in views.items()}
    for k, _ in KINDS:
        setattr(f, k, fields[k])
    api.FreeFramebuffer(fb)
    del busy
    for k, _ in KINDS:
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("replaced", [("color",), ("depth", "stencil"), ("color", "depth", "stencil")])
def test_freeing_leaves_the_callers_arrays_alone(api, replaced):
    """A framebuffer freed with the program's own arrays in place of some or
    all of its own: they keep what the last download wrote, and the program's
    next framebuffer works."""
    w, h = 67, 61
    mine = {k: np.zeros(w * h * n, np.uint8) for k, n in KINDS}
    want = {}
    for turn in range(2):
        fb = api.NewFramebuffer(w, h)
        f = api.Fields.from_address(fb)
        for k in replaced:
            setattr(f, k, mine[k].ctypes.data)
        rng = np.random.default_rng(turn)
        views = host_arrays(api, fb)
        for k, v in views.items():
            v[:] = want[k] = rng.integers(0, 256, v.size, dtype=np.uint8)
        api.FramebufferSetDeferred(fb, True)
        for v in views.values():
            v[:] = 0
        api.FramebufferDownload(fb)
        del views
        api.FreeFramebuffer(fb)
        for k in replaced:
            assert np.array_equal(mine[k], want[k]), k
            mine[k][:] = 7


def test_staged_passes_keep_the_colours_of_their_call(api):
    """The five passes of a synchronous framebuffer, each cleared (on the
    host) as soon as it is staged."""
    w, h = 640, 360
    n = w * h
    fb = api.NewFramebuffer(w, h)
    views = host_arrays(api, fb)
    rng = np.random.default_rng(2)
    passes = rng.integers(0, 1 << 32, (5, n), dtype=np.uint32)
    dataset = api.NewNeuralDataset(n)
    api.FramebufferClear(fb)
    busy = keep_busy(api)
    for k in range(5):
        views["color"][:] = passes[k].view(np.uint8)
        api.NeuralDatasetStage(dataset, fb, k)
        api.FramebufferClear(fb)
    api.FramebufferFillDepth(fb, 0.5)
    count = api.NeuralDatasetAppend(dataset, fb, 1.0, 3)
    features, targets = np.empty((n, 8), np.float32), np.empty((n, 3), np.float32)
    if count == n:
        api.NeuralDatasetRead(dataset, 0, n, features.ctypes.data, targets.ctypes.data)
    api.FreeNeuralDataset(dataset)
    api.FreeFramebuffer(fb)
    del busy
    assert count == n
    f = np.empty((n, 8), np.float32)
    for k in range(4):
        f[:, 2 * k] = (passes[k] >> 16).astype(np.float32) / np.float32(65535)
        f[:, 2 * k + 1] = (passes[k] & 0xFFFF).astype(np.float32) / np.float32(65535)
    f[:, 3:6] = f[:, 3:6] * np.float32(2) - np.float32(1)
    t = np.stack([(passes[4] >> s & 255).astype(np.float32) / np.float32(255) for s in (24, 16, 8)], -1)
    assert np.array_equal(features, f)
    assert np.array_equal(targets, t)
