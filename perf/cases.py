"""The work this renderer is measured on: frames, batches, G-buffer capture and
the learned shader's training and inference, each through the C API of
include/srp (srp.h, srp_hip.h, srp_neural.h) as a host program calls it, with
the device shaders of the repository's scene module.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)`
one more of the same ranges, `prepare(case, seed)` what a program holds before
the call, `run(state)` one pass and its outputs, `work(case)` the bytes and
operations of a pass, `exact(case, seed)` the outputs in 64 bits where a closed
formula gives them.

Frames end in `srpFramebufferDownload` (or in a synchronous draw): the host
arrays of SRPFramebuffer are where this API delivers its result.
"""
import ctypes as C
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# enum values of include/srp/{context,buffer,type,vertex,texture}.h
FACE_BACK = 2
CMP_ALWAYS, CMP_LESS, CMP_LEQUAL, CMP_GREATER = 1, 2, 3, 4
ST_KEEP, ST_INCR = 0, 3
PRIM_POINTS, PRIM_LINES, PRIM_TRIANGLES = 0, 1, 4
T_FLOAT, T_UINT8, T_UINT16, T_UINT32 = 0, 6, 7, 8
PERSPECTIVE, AFFINE, FLAT = 0, 1, 2
MODES = {"fill": 0, "line": 1, "point": 2}

vp, sz, i32, u8, u32, u64, f32, b1 = C.c_void_p, C.c_size_t, C.c_int, C.c_uint8, C.c_uint32, C.c_uint64, C.c_float, C.c_bool


class Framebuffer(C.Structure):
    _fields_ = [("width", sz), ("height", sz), ("size", sz), ("color", vp), ("depth", vp), ("stencil", vp)]


class VaryingInfo(C.Structure):
    _fields_ = [("nItems", sz), ("type", i32), ("mode", i32)]


class VertexShader(C.Structure):
    _fields_ = [("shader", vp), ("nVaryings", sz), ("varyingsInfo", C.POINTER(VaryingInfo)), ("varyingsSize", sz)]


class FragmentShader(C.Structure):
    _fields_ = [("shader", vp), ("mayOverwriteDepth", b1)]


class Program(C.Structure):
    _fields_ = [("uniform", vp), ("vs", C.POINTER(VertexShader)), ("fs", C.POINTER(FragmentShader))]


class UniTexture(C.Structure):
    _fields_ = [("frame", u64), ("model", f32 * 16), ("view", f32 * 16), ("projection", f32 * 16), ("texture", vp)]


class UniMVP(C.Structure):
    _fields_ = [("model", f32 * 16), ("view", f32 * 16), ("projection", f32 * 16)]


class UniTerrain(C.Structure):
    _fields_ = [("viewProj", f32 * 16), ("lo", f32 * 3), ("inv", f32 * 3), ("capture", u32), ("pad", u32), ("network", vp)]


class DrawCommand(C.Structure):
    _fields_ = [("ib", vp), ("vb", vp), ("fb", vp), ("sp", C.POINTER(Program)), ("primitive", i32), ("startIndex", sz),
                ("count", sz), ("context", vp), ("clear", i32), ("clearDepth", f32), ("clearStencil", u8)]


class BatchTuning(C.Structure):
    _fields_ = [(n, i32) for n in ("wavesPerCU", "maskBox", "xcdQueues", "pixelRuns", "depthCull", "tileSize")]


SIGNATURES = {
    "srpNewContext": (None, [vp]), "srpScissorTest": (None, [b1]), "srpScissorOptions": (None, [sz] * 4),
    "srpStencilTest": (None, [b1]), "srpStencilFunc": (None, [i32, u8, u8]), "srpStencilOp": (None, [i32] * 3),
    "srpDepthTest": (None, [b1]), "srpDepthCompareOp": (None, [i32]), "srpRasterCullFace": (None, [i32]),
    "srpRasterPolygonMode": (None, [i32]), "srpRasterPointSize": (None, [f32]),
    "srpNewVertexBuffer": (vp, []), "srpFreeVertexBuffer": (None, [vp]),
    "srpVertexBufferCopyData": (None, [vp, sz, sz, vp]),
    "srpNewIndexBuffer": (vp, []), "srpFreeIndexBuffer": (None, [vp]), "srpIndexBufferCopyData": (None, [vp, i32, sz, vp]),
    "srpDrawVertexBuffer": (None, [vp, vp, vp, i32, sz, sz]), "srpDrawIndexBuffer": (None, [vp, vp, vp, vp, i32, sz, sz]),
    "srpNewFramebuffer": (vp, [sz, sz]), "srpFreeFramebuffer": (None, [vp]), "srpFramebufferClear": (None, [vp]),
    "srpFramebufferSetDeferred": (None, [vp, b1]), "srpFramebufferDownload": (None, [vp]),
    "srpFramebufferFillDepth": (None, [vp, f32]), "srpFramebufferFillStencil": (None, [vp, u8]),
    "srpNewTextureFromMemory": (vp, [vp, i32, i32, i32, i32]), "srpFreeTexture": (None, [vp]),
    "srpNewBatch": (vp, [vp, sz]), "srpFreeBatch": (None, [vp]), "srpBatchRender": (None, [vp]),
    "srpBatchCapture": (i32, [vp]), "srpBatchSetTuning": (None, [vp, vp]), "srpBatchGetTuning": (None, [vp, vp]),
    "srpNewNeuralDataset": (vp, [sz]), "srpFreeNeuralDataset": (None, [vp]),
    "srpNeuralDatasetStage": (None, [vp, vp, i32]), "srpNeuralDatasetAppend": (sz, [vp, vp, f32, u64]),
    "srpNeuralDatasetRead": (None, [vp, sz, sz, vp, vp]), "srpNeuralDatasetWrite": (None, [vp, vp, vp, sz]),
    "srpNewNeuralNet": (vp, [u64]), "srpFreeNeuralNet": (None, [vp]), "srpNeuralNetSetParams": (None, [vp, vp]),
    "srpNeuralNetGetParams": (None, [vp, vp]), "srpNeuralNetSetEncoding": (None, [vp, vp]),
    "srpNeuralNetTrain": (None, [vp, vp, i32, i32, f32, f32, u64, vp]),
    "srpNeuralNetInfer": (None, [vp, vp, sz, vp, i32]), "srpNeuralNetDevice": (vp, [vp]),
}

_api = None


class Api:
    """The library, the scene module whose shaders the programs name, and the
    program's one context."""

    def __init__(self):
        lib = C.CDLL(os.path.join(ROOT, "srp_amd", "libsrp_amd.so"))
        scenes = C.CDLL(os.path.join(ROOT, "tests", "scenes", "build", "libscenes_amd.so"))
        for name, (res, args) in SIGNATURES.items():
            f = getattr(lib, name)
            f.restype, f.argtypes = res, args
            setattr(self, name[3:], f)
        self.shader = lambda name: C.cast(getattr(scenes, name), vp).value
        self.context = C.create_string_buffer(256)
        self.NewContext(self.context)

    def program(self, vs, varyings, fs, uniform=None):
        info = (VaryingInfo * len(varyings))(*[VaryingInfo(*v) for v in varyings])
        V = VertexShader(self.shader(vs), len(varyings), info, 4 * sum(v[0] for v in varyings))
        F = FragmentShader(self.shader(fs), False)
        P = Program(C.addressof(uniform) if uniform is not None else None, C.pointer(V), C.pointer(F))
        P.keep = (info, V, F, uniform)
        return P


def api():
    global _api
    if _api is None:
        _api = Api()
    return _api


class State:
    """What a program keeps between frames; freed through the API."""

    def __init__(self, kind):
        self.kind, self.owned = kind, []

    def own(self, free, handle):
        if not handle:
            raise RuntimeError("the library made no %s" % free)
        self.owned.append((free, handle))
        return handle

    def __del__(self):
        for free, handle in reversed(self.owned):
            getattr(api(), free)(handle)

    def vertices(self, array, stride):
        a = api()
        b = self.own("FreeVertexBuffer", a.NewVertexBuffer())
        a.VertexBufferCopyData(b, stride, array.nbytes, array.ctypes.data)
        return b

    def indices(self, array):
        a = api()
        b = self.own("FreeIndexBuffer", a.NewIndexBuffer())
        a.IndexBufferCopyData(b, {1: T_UINT8, 2: T_UINT16, 4: T_UINT32}[array.itemsize], array.nbytes, array.ctypes.data)
        return b

    def framebuffer(self, w, h, deferred=True):
        a = api()
        target = Target(w, h)
        self.images = target.images()
        if deferred:
            a.FramebufferSetDeferred(target.fb, True)
        return target.fb

    def save_context(self):
        """The render state set since srpNewContext, as the program restores it."""
        self.context = api().context.raw

    def use_context(self):
        C.memmove(api().context, self.context, len(self.context))


class Target:
    """A framebuffer, freed with the last array that shows its pixels."""

    def __init__(self, w, h):
        self.fb = api().NewFramebuffer(w, h)

    def __del__(self):
        api().FreeFramebuffer(self.fb)

    def images(self):
        """The host arrays of the framebuffer (colour as int32 bits)."""
        f = Framebuffer.from_address(self.fb)

        def arr(p, t, dt):
            pixels = (t * f.size).from_address(p)
            pixels.target = self
            return np.ndarray(f.size, dt, pixels)

        return [arr(f.color, C.c_int32, np.int32), arr(f.depth, f32, np.float32), arr(f.stencil, u8, np.uint8)]


def start_frame(a, fb, depth=1.0, stencil=0):
    a.FramebufferClear(fb)
    a.FramebufferFillDepth(fb, depth)
    a.FramebufferFillStencil(fb, stencil)


# ---------------------------------------------------------------- matrices

def perspective(aspect, fov_deg, near, far):
    """mat4ConstructPerspectiveProjection of a symmetric frustum."""
    t = math.tan(math.radians(fov_deg) / 2)
    return np.array([[1 / (t * aspect), 0, 0, 0], [0, 1 / t, 0, 0],
                     [0, 0, (far + near) / (far - near), -2 * near * far / (far - near)], [0, 0, 1, 0]])


def rotation(x, y, z):
    sx, cx, sy, cy, s, c = math.sin(x), math.cos(x), math.sin(y), math.cos(y), math.sin(z), math.cos(z)
    return np.array([[cy * c, sx * sy * c - cx * s, cx * sy * c + sx * s], [cy * s, sx * sy * s + cx * c, cx * sy * s - sx * c],
                     [-sy, sx * cy, cx * cy]])


def placed(position, angles, scale):
    m = np.eye(4)
    m[:3, :3] = rotation(*angles) * scale
    m[:3, 3] = position
    return m


def look(eye, forward):
    r = np.array([forward[2], 0, -forward[0]])
    r /= np.linalg.norm(r)
    up = np.cross(forward, r)
    m = np.eye(4)
    m[:3, :3] = [r, up, forward]
    m[:3, 3] = -m[:3, :3] @ np.asarray(eye)
    return m


def mat(m):
    return (f32 * 16)(*np.asarray(m, np.float32).ravel().tolist())


# ---------------------------------------------------------------- geometry

def sphere(rings, segs):
    """UV sphere {position, uv}, indexed triangles (degenerate at the poles)."""
    i, j = np.meshgrid(np.arange(rings + 1), np.arange(segs + 1), indexing="ij")
    th, ph = np.pi * i / rings, 2 * np.pi * j / segs
    v = np.stack([np.sin(th) * np.cos(ph), np.cos(th), np.sin(th) * np.sin(ph), j / segs, 1 - i / rings], -1)
    q = (np.arange(rings)[:, None] * (segs + 1) + np.arange(segs)[None]).ravel()
    r = q + segs + 1
    idx = np.stack([q, r, q + 1, r, r + 1, q + 1], -1)
    return v.reshape(-1, 5).astype(np.float32), idx.ravel()


def cube():
    """24 vertices {position, uv}, 36 indices."""
    v, idx = [], []
    for axis in range(3):
        for side in (-1.0, 1.0):
            for s, t in ((-1, -1), (1, -1), (1, 1), (-1, 1)):
                p = [0.0, 0.0, 0.0]
                p[axis], p[(axis + 1) % 3], p[(axis + 2) % 3] = side, s * side, t
                v.append(p + [(s + 1) / 2, (t + 1) / 2])
            k = len(v) - 4
            idx += [k, k + 1, k + 2, k, k + 2, k + 3]
    return np.array(v, np.float32) * np.array([0.6, 0.6, 0.6, 1, 1], np.float32), np.array(idx)


def heightfield(nx, nz, seed):
    """Rolling terrain over x in [-10, 10], z in [-5, 5]: {position, normal,
    uv}, indexed triangles, and the height function's waves."""
    rng = np.random.default_rng(seed)
    k = rng.normal(0, 1, (28, 2)) * (0.35 * 1.17 ** np.arange(28))[:, None]
    amp = 0.75 / (1 + np.linalg.norm(k, axis=1)) ** 1.6
    phase = rng.uniform(0, 2 * np.pi, 28)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.linspace(-10, 10, nx + 1, dtype=torch.float64, device=dev)
    z = torch.linspace(-5, 5, nz + 1, dtype=torch.float64, device=dev)
    zz, xx = torch.meshgrid(z, x, indexing="ij")
    h, hx, hz = (torch.zeros_like(xx) for _ in range(3))
    for (kx, kz), a, p in zip(k.tolist(), amp.tolist(), phase.tolist()):
        t = kx * xx + kz * zz + p
        h += a * torch.sin(t)
        c = a * torch.cos(t)
        hx += kx * c
        hz += kz * c
    n = torch.sqrt(hx * hx + 1 + hz * hz)
    u, w = torch.meshgrid(torch.linspace(0, 1, nz + 1, device=dev), torch.linspace(0, 1, nx + 1, device=dev), indexing="ij")
    v = torch.stack([xx, h, zz, -hx / n, 1 / n, -hz / n, w, u], -1).float().reshape(-1, 8).cpu().numpy()
    a = (np.arange(nz)[:, None] * (nx + 1) + np.arange(nx)[None]).ravel()
    c = a + nx + 1
    idx = np.stack([a, a + 1, c, a + 1, c + 1, c], -1).ravel().astype(np.uint32)
    return v, idx, (float(h.min()), float(h.max())), lambda px, pz: float(np.sum(amp * np.sin(k @ [px, pz] + phase)))


MIX_VERTEX = np.dtype([("clip", "f4", 4), ("st", "f4", 2), ("level", "f4"), ("tag", "u4")])


def mix_vertices(rng, xy, z, w):
    v = np.empty(xy.shape[:-1], MIX_VERTEX)
    v["clip"] = np.concatenate([xy * w[..., None], (z * w)[..., None], w[..., None]], -1)
    v["st"] = rng.random(v.shape + (2,))
    v["level"] = rng.random(v.shape)
    v["tag"] = rng.integers(0, 1 << 32, v.shape, dtype=np.uint32)
    return v.ravel()


def mix_triangles(rng, n):
    """Clip-space triangles of lognormal size; three in ten reach behind the
    near plane, one in ten lies outside."""
    c, size = rng.uniform(-1, 1, (n, 1, 2)), np.exp(-3 + rng.normal(size=(n, 1)))
    ang = 2 * np.pi * rng.random((n, 1)) + np.arange(3) * (2 * np.pi / 3) + 0.3 * rng.random((n, 3))
    kind = rng.random((n, 1))
    xy = c + size[..., None] * np.stack([np.cos(ang), np.sin(ang)], -1)
    z = rng.uniform(-0.9, 0.9, (n, 1)) + rng.uniform(-0.05, 0.05, (n, 3))
    behind = (kind < 0.3) & (np.arange(3) < 1 + (kind * 10).astype(int) % 2)
    z = np.where(behind, rng.uniform(-3, -1.2, (n, 3)), z)
    xy[..., 0] += np.where((kind >= 0.3) & (kind < 0.4), 3.5, 0.0)
    return mix_vertices(rng, xy, z, rng.uniform(0.6, 1.6, (n, 3)))


def mix_lines(rng, n):
    c, size, ang = rng.uniform(-1.1, 1.1, (n, 1, 2)), np.exp(-2.5 + 0.7 * rng.normal(size=(n, 1))), 2 * np.pi * rng.random((n, 1))
    s = np.array([-0.5, 0.5]) * size
    xy = c + np.stack([s * np.cos(ang), s * np.sin(ang)], -1)
    return mix_vertices(rng, xy, rng.uniform(-1.1, 1.1, (n, 2)), rng.uniform(0.8, 1.2, (n, 2)))


def mix_points(rng, n):
    return mix_vertices(rng, rng.uniform(-1.05, 1.05, (n, 2)), rng.uniform(-1, 1, n), rng.uniform(0.8, 1.2, n))


# ------------------------------------------------------------------- cases

def listed():
    return [
        # One textured cube in a small window, default (synchronous) mode: what
        # a program written for the reference does each frame; latency counts.
        {"name": "cube_sync", "kind": "objects", "w": 256, "h": 256, "objects": 1, "rings": 0, "segs": 0, "index": 1,
         "mode": "fill", "sync": True, "texture": 64},
        # A wireframe model at the reference's test size, synchronous.
        {"name": "wireframe_sync", "kind": "objects", "w": 512, "h": 512, "objects": 1, "rings": 24, "segs": 48, "index": 2,
         "mode": "line", "sync": True, "texture": 64},
        # Few large overlapping triangles: fill and depth complexity.
        {"name": "triangles_512", "kind": "triangles", "w": 512, "h": 512, "n": 2000},
        # A scene of many small objects: one short draw each.
        {"name": "objects_720p", "kind": "objects", "w": 1280, "h": 720, "objects": 96, "rings": 12, "segs": 24, "index": 2,
         "mode": "fill", "sync": False, "texture": 256},
        # Eight dense textured meshes (262,144 triangles each) in a 1080p frame.
        {"name": "mesh_1080p", "kind": "objects", "w": 1920, "h": 1080, "objects": 8, "rings": 256, "segs": 512, "index": 4,
         "mode": "fill", "sync": False, "texture": 1024},
        # The primitive mix: clipped triangles of every size, lines, points.
        {"name": "mix_1080p", "kind": "mix", "w": 1920, "h": 1080, "triangles": 500000, "lines": 100000, "points": 100000},
        # A million-triangle terrain with the expensive procedural material,
        # camera inside it, so that triangles are clipped.
        {"name": "terrain_1080p", "kind": "terrain", "w": 1920, "h": 1080, "nx": 1000, "nz": 500, "neural": False, "views": 1},
        # The same with the learned material on the matrix cores.
        {"name": "terrain_neural_1080p", "kind": "terrain", "w": 1920, "h": 1080, "nx": 1000, "nz": 500, "neural": True, "views": 1},
        # Independent scenes, each with its own camera, state and framebuffer,
        # rendered as one captured batch.
        {"name": "batch_20", "kind": "batch", "scenes": 20, "side": 768, "triangles": 60000, "waves": 28},
        # Collecting the learned shader's training data: one pose of four
        # G-buffer passes and the shaded frame, decoded into samples.
        {"name": "capture_1080p", "kind": "capture", "w": 1920, "h": 1080, "nx": 1000, "nz": 500, "keep": 0.0135},
        # Training the learned shader, at the batch the benchmark trains with.
        {"name": "train_8192", "kind": "train", "samples": 262144, "batch": 8192, "steps": 32},
        # The network alone over a frame's worth of samples and more.
        {"name": "infer_1m", "kind": "infer", "samples": 1048576},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["objects", "objects", "objects", "triangles", "mix", "terrain", "batch", "capture", "train", "infer"])
    w = log_int(160, 1920)
    h = max(120, min(1080, int(w * rng.uniform(0.5, 1.0))))
    if kind == "objects":
        rings = log_int(3, 256)
        n = min(64, max(1, int(log_int(2000, 1500000) / (4 * rings * rings))))
        sync = n <= 4 and rng.random() < 0.5
        mode = rng.choice(["fill", "fill", "fill", "line", "point"]) if rings <= 64 else "fill"
        verts = (rings + 1) * (2 * rings + 1)
        return {"kind": kind, "w": w, "h": h, "objects": n, "rings": rings, "segs": 2 * rings,
                "index": 1 if verts <= 255 else 2 if verts <= 65535 else 4, "mode": mode, "sync": sync,
                "texture": log_int(16, 1024)}
    if kind == "triangles":
        return {"kind": kind, "w": min(w, 1024), "h": min(h, 1024), "n": log_int(1, 2500)}
    if kind == "mix":
        n = log_int(500, 250000)
        return {"kind": kind, "w": w, "h": h, "triangles": n, "lines": n // 5 + rng.randrange(9),
                "points": n // 5 + rng.randrange(9)}
    if kind in ("terrain", "capture"):
        nx = log_int(40, 1000)
        c = {"kind": kind, "w": w, "h": h, "nx": nx, "nz": max(20, nx // 2 + rng.randrange(7))}
        return {**c, "neural": rng.random() < 0.4, "views": rng.randint(1, 4)} if kind == "terrain" else {**c, "keep": rng.uniform(0.005, 1.0)}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 20), "side": log_int(64, 768), "triangles": log_int(50, 60000),
                "waves": rng.choice([8, 16, 28])}
    if kind == "train":
        return {"kind": kind, "samples": log_int(1500, 262144), "batch": 1024 * log_int(1, 16), "steps": rng.randint(2, 32)}
    return {"kind": kind, "samples": log_int(50, 1048576)}


# ----------------------------------------------------------------- prepare

def prepare(case, seed):
    a = api()
    s = State(case["kind"])
    s.case = case
    a.NewContext(a.context)
    globals()["prepare_" + case["kind"]](a, s, case, np.random.default_rng(seed), seed)
    s.save_context()
    return s


def prepare_objects(a, s, case, rng, seed):
    """Textured objects spread over the view, each with its own transform;
    scissor, stencil and depth as the textured-mesh workload sets them."""
    w, h = case["w"], case["h"]
    v, idx = sphere(case["rings"], case["segs"]) if case["rings"] else cube()
    s.vb = s.vertices(v, 20)
    s.ib = s.indices(np.ascontiguousarray(idx.astype({1: np.uint8, 2: np.uint16, 4: np.uint32}[case["index"]])))
    s.count = len(idx)
    t = case["texture"]
    texels = rng.integers(0, 256, (t, t, 3), dtype=np.uint8)
    texture = s.own("FreeTexture", a.NewTextureFromMemory(texels.ctypes.data, t, t, 0, 0))
    n = case["objects"]
    side = math.ceil(math.sqrt(n))
    proj, view = mat(perspective(w / h, 60, 0.1, 100)), mat(np.eye(4))
    s.programs = []
    for k in range(n):
        # a jittered grid over the screen, so that the frame's coverage is alike for every seed
        z = 2.6 * (1 + 0.75 * (side - 1)) * rng.uniform(0.9, 1.1)
        x = ((k % side + 0.5) / side * 2 - 1) * (1 - 1 / side) * z * 0.5 * w / h + rng.uniform(-0.1, 0.1)
        y = ((k // side + 0.5) / side * 2 - 1) * (1 - 1 / side) * z * 0.5 + rng.uniform(-0.1, 0.1)
        u = UniTexture(k, mat(placed((x, y, z), rng.uniform(0, 6.28, 3), 1.0)), view, proj, texture)
        s.programs.append(a.program("sc_vsMeshTex", [(2, T_FLOAT, PERSPECTIVE), (1, T_UINT32, FLAT)], "sc_fsMeshTex", u))
    s.fb = s.framebuffer(w, h, not case["sync"])
    a.ScissorTest(True)
    a.ScissorOptions(w // 16, h // 16, w * 7 // 8, h * 7 // 8)
    a.StencilTest(True)
    a.StencilFunc(CMP_ALWAYS, 0, 0xFF)
    a.StencilOp(ST_KEEP, ST_KEEP, ST_INCR)
    a.DepthTest(True)
    a.DepthCompareOp(CMP_LESS)
    a.RasterPolygonMode(MODES[case["mode"]])
    a.RasterPointSize(2.0)


def prepare_triangles(a, s, case, rng, seed):
    """Random clip-space triangles with a colour per vertex."""
    v = np.concatenate([rng.uniform(-1.2, 1.2, (3 * case["n"], 3)), rng.random((3 * case["n"], 3))], -1).astype(np.float32)
    s.vb = s.vertices(v, 24)
    s.program = a.program("sc_vsColorPass", [(3, T_FLOAT, PERSPECTIVE)], "sc_fsColor")
    s.fb = s.framebuffer(case["w"], case["h"])
    a.DepthTest(True)
    a.DepthCompareOp(CMP_LESS)


def prepare_mix(a, s, case, rng, seed):
    s.vbs = [s.vertices(f(rng, n), 32) for f, n in
             ((mix_triangles, case["triangles"]), (mix_lines, case["lines"]), (mix_points, case["points"]))]
    s.program = a.program("sc_vsMix", [(2, T_FLOAT, AFFINE), (1, T_FLOAT, FLAT), (1, T_UINT32, FLAT)], "sc_fsMix")
    s.fb = s.framebuffer(case["w"], case["h"])
    a.DepthTest(True)
    a.DepthCompareOp(CMP_LEQUAL)
    a.RasterCullFace(FACE_BACK)


def make_terrain(a, s, case, rng, seed, fs, capture=0, network=None, pose=0):
    if pose == 0:
        s.fbs, s.outputs = [], []
        v, idx, (lo, hi), s.height = heightfield(case["nx"], case["nz"], seed)
        s.vb, s.ib, s.count, s.range = s.vertices(v, 32), s.indices(idx), len(idx), (lo, hi)
    s.fbs.append(s.framebuffer(case["w"], case["h"]))
    s.outputs.append(s.images)
    lo, hi = s.range
    yaw, pitch = rng.uniform(0, 2 * math.pi), math.radians(rng.uniform(25, 40))
    ex, ez = rng.uniform(-6, 6), rng.uniform(-3, 3)
    forward = np.array([math.cos(pitch) * math.cos(yaw), -math.sin(pitch), math.cos(pitch) * math.sin(yaw)])
    eye = (ex, s.height(ex, ez) + rng.uniform(1.5, 3.0), ez)
    vpm = perspective(case["w"] / case["h"], 60, 0.1, 100) @ look(eye, forward)
    u = UniTerrain(mat(vpm), (f32 * 3)(-10, lo, -5), (f32 * 3)(0.05, 1 / (hi - lo), 0.1), capture, 0, network)
    return a.program("sc_vsTerrain", [(3, T_FLOAT, PERSPECTIVE), (3, T_FLOAT, PERSPECTIVE), (2, T_FLOAT, PERSPECTIVE)], fs, u)


def terrain_state(a):
    a.DepthTest(True)
    a.DepthCompareOp(CMP_LESS)
    a.RasterCullFace(FACE_BACK)


def prepare_terrain(a, s, case, rng, seed):
    """Views of the terrain, each in a framebuffer of its own."""
    network = None
    if case["neural"]:
        s.net = make_net(a, s, rng)[0]
        network = a.NeuralNetDevice(s.net)
    fs = "sc_fsTerrainNeural" if case["neural"] else "sc_fsTerrain"
    s.programs = [make_terrain(a, s, case, rng, seed, fs, 0, network, k) for k in range(case["views"])]
    terrain_state(a)


def prepare_capture(a, s, case, rng, seed):
    first = make_terrain(a, s, case, rng, seed, "sc_fsTerrain")
    u = first.keep[3]
    s.programs = []
    for k in range(4):
        uk = UniTerrain(u.viewProj, u.lo, u.inv, k, 0, None)
        s.programs.append(a.program("sc_vsTerrain", [(3, T_FLOAT, PERSPECTIVE), (3, T_FLOAT, PERSPECTIVE), (2, T_FLOAT, PERSPECTIVE)],
                                    "sc_fsTerrainCapture", uk))
    s.programs.append(first)
    s.seed = seed
    cap = int(case["w"] * case["h"] * case["keep"]) + 1024
    s.fb = s.fbs[0]
    s.dataset = s.own("FreeNeuralDataset", a.NewNeuralDataset(cap))
    s.features, s.targets = np.zeros((cap, 8), np.float32), np.zeros((cap, 3), np.float32)
    terrain_state(a)


def prepare_batch(a, s, case, rng, seed):
    """Triangle soups, each seen by its own camera into its own framebuffer,
    with sides and triangle counts spread below the case's."""
    n = case["scenes"]
    info = [(3, T_FLOAT, PERSPECTIVE)]
    cmds = (DrawCommand * n)()
    s.fbs, s.outputs, s.programs, s.contexts = [], [], [], []
    sides = [max(16, int(case["side"] * f)) for f in np.linspace(0.2, 1.0, n)]
    counts = [max(1, int(case["triangles"] * f)) for f in rng.permutation(np.linspace(0.1, 1.9, n) ** 2)]
    V = FS = None
    for k, (side, m) in enumerate(zip(sides, counts)):
        d = rng.normal(size=3) * [1, 0.5, 1]
        d /= np.linalg.norm(d)
        u = UniMVP(mat(np.eye(4)), mat(look(d * rng.uniform(2.6, 4.2), -d)), mat(perspective(1.0, rng.uniform(50, 70), 0.1, 20)))
        p = a.program("sc_vsColorMVP", info, "sc_fsColor", u)
        if V is None:
            V, FS = p.vs, p.fs
        p.vs, p.fs = V, FS
        s.programs.append(p)
        centre, size = rng.uniform(-1, 1, (m, 1, 3)), np.exp(math.log(0.05) + 0.6 * rng.normal(size=(m, 1, 1)))
        v = np.concatenate([centre + size * rng.uniform(-1, 1, (m, 3, 3)), rng.random((m, 3, 3))], -1).astype(np.float32)
        a.NewContext(a.context)
        a.DepthTest(True)
        a.DepthCompareOp(CMP_GREATER if k % 5 == 4 else CMP_LESS)
        if k % 3 == 1:
            a.RasterCullFace(FACE_BACK)
        if k % 4 == 3:
            a.StencilTest(True)
            a.StencilOp(ST_KEEP, ST_KEEP, ST_INCR)
        s.contexts.append(C.create_string_buffer(a.context.raw, 256))
        s.fbs.append(s.framebuffer(side, side))
        s.outputs.append(s.images)
        cmds[k] = DrawCommand(None, s.vertices(v, 24), s.fbs[-1], C.pointer(p), PRIM_TRIANGLES, 0, 3 * m,
                              C.addressof(s.contexts[-1]), 1, -1.0 if k % 5 == 4 else 1.0, 0)
    s.cmds = cmds
    s.batch = s.own("FreeBatch", a.NewBatch(cmds, n))
    a.BatchSetTuning(s.batch, C.byref(BatchTuning(case["waves"], 24, 1, 1, 1, 8)))
    if a.BatchCapture(s.batch) != 0:
        raise RuntimeError("the batch could not be captured")


NN_PARAMS = 37187
NN_STEPS = np.array([1.0, 0.5, 0.75, 0.5, 0.5, 0.5, 2.0, 1.0], np.float32)


def net_params(rng):
    """Weights and biases uniform in +-1/sqrt(fan in), the library's layout."""
    fan = np.full(NN_PARAMS, 64.0)
    fan[:64 * 512 + 64] = 512.0
    return (rng.uniform(-1, 1, NN_PARAMS) / np.sqrt(fan)).astype(np.float32)


def make_net(a, s, rng):
    net = s.own("FreeNeuralNet", a.NewNeuralNet(1))
    p = net_params(rng)
    a.NeuralNetSetParams(net, p.ctypes.data)
    a.NeuralNetSetEncoding(net, NN_STEPS.ctypes.data)
    return net, p


def samples(rng, n):
    """Surface features (position and UV in [0, 1], unit normals pointing up)
    and the smooth colours a material gives them."""
    x = rng.random((n, 8))
    nrm = rng.normal(0, 0.4, (n, 3)) + [0, 1, 0]
    x[:, 3:6] = nrm / np.linalg.norm(nrm, axis=1, keepdims=True)
    light = np.clip(x[:, 3:6] @ [0.27, 0.8, 0.53], 0, 1)[:, None]
    t = (0.15 + 0.7 * light) * (0.5 + 0.3 * np.sin(2 * np.pi * (x[:, [0, 1, 2]] * [2, 1, 3] + x[:, [2, 0, 1]])))
    return np.ascontiguousarray(x, np.float32), np.ascontiguousarray(t, np.float32)


def make_samples(a, s, rng, n):
    x, t = samples(rng, n)
    ds = s.own("FreeNeuralDataset", a.NewNeuralDataset(n))
    a.NeuralDatasetWrite(ds, x.ctypes.data, t.ctypes.data, n)
    return ds


def prepare_train(a, s, case, rng, seed):
    s.net, _ = make_net(a, s, rng)
    s.dataset = make_samples(a, s, rng, case["samples"])
    s.params, s.loss = np.empty(NN_PARAMS, np.float32), np.empty(case["steps"], np.float32)


TRAIN_LR = (1e-4, 2e-6)
TRAIN_SEED = 0x5EED0005


def prepare_infer(a, s, case, rng, seed):
    s.net, _ = make_net(a, s, rng)
    s.dataset = make_samples(a, s, rng, case["samples"])
    pin = torch.cuda.is_available()
    s.rgb = torch.empty((case["samples"], 3), dtype=torch.float32, pin_memory=pin)


# --------------------------------------------------------------------- run

def run(s):
    return globals()["run_" + s.kind](api(), s, s.case)


def run_objects(a, s, case):
    s.use_context()
    fb = s.fb
    start_frame(a, fb)
    for p in s.programs:
        a.DrawIndexBuffer(s.ib, s.vb, fb, C.byref(p), PRIM_TRIANGLES, 0, s.count)
    if not case["sync"]:
        a.FramebufferDownload(fb)
    return s.images


def run_triangles(a, s, case):
    s.use_context()
    start_frame(a, s.fb)
    a.DrawVertexBuffer(s.vb, s.fb, C.byref(s.program), PRIM_TRIANGLES, 0, 3 * case["n"])
    a.FramebufferDownload(s.fb)
    return s.images


def run_mix(a, s, case):
    s.use_context()
    fb, p = s.fb, C.byref(s.program)
    start_frame(a, fb)
    a.DrawVertexBuffer(s.vbs[0], fb, p, PRIM_TRIANGLES, 0, 3 * case["triangles"])
    a.DrawVertexBuffer(s.vbs[1], fb, p, PRIM_LINES, 0, 2 * case["lines"])
    q = case["points"] // 4
    for k in range(4):
        a.RasterPointSize(float(k + 1))
        a.DrawVertexBuffer(s.vbs[2], fb, p, PRIM_POINTS, k * q, q)
    a.FramebufferDownload(fb)
    return s.images


def run_terrain(a, s, case):
    s.use_context()
    for fb, p in zip(s.fbs, s.programs):
        start_frame(a, fb)
        a.DrawIndexBuffer(s.ib, s.vb, fb, C.byref(p), PRIM_TRIANGLES, 0, s.count)
    for fb in s.fbs:
        a.FramebufferDownload(fb)
    return s.outputs


def run_batch(a, s, case):
    a.BatchRender(s.batch)
    for fb in s.fbs:
        a.FramebufferDownload(fb)
    return s.outputs


def run_capture(a, s, case):
    s.use_context()
    a.NeuralDatasetWrite(s.dataset, s.features.ctypes.data, s.targets.ctypes.data, 0)
    for k, p in enumerate(s.programs):
        start_frame(a, s.fb)
        a.DrawIndexBuffer(s.ib, s.vb, s.fb, C.byref(p), PRIM_TRIANGLES, 0, s.count)
        a.NeuralDatasetStage(s.dataset, s.fb, k)
    n = a.NeuralDatasetAppend(s.dataset, s.fb, case["keep"], s.seed)
    a.NeuralDatasetRead(s.dataset, 0, n, s.features.ctypes.data, s.targets.ctypes.data)
    return [s.features, s.targets, n]


def run_train(a, s, case):
    a.NeuralNetTrain(s.net, s.dataset, case["steps"], case["batch"], *TRAIN_LR, TRAIN_SEED, s.loss.ctypes.data)
    a.NeuralNetGetParams(s.net, s.params.ctypes.data)
    return {"params": s.params, "loss": s.loss}


def run_infer(a, s, case):
    a.NeuralNetInfer(s.net, s.dataset, case["samples"], s.rgb.data_ptr(), 0)
    return s.rgb


# -------------------------------------------------------------------- work

NN_FORWARD = 2 * (512 * 64 + 64 * 64 + 64 * 3)
NN_TRAIN = 3 * NN_FORWARD - 2 * 512 * 64   # no gradient of the encoded input
SHADE_TERRAIN = 2800   # operations of the procedural material per fragment


def work(case):
    k = case["kind"]
    if k == "train":
        # per step: its samples, and parameters and their two moments read and written once
        return {"bytes": case["steps"] * (case["batch"] * 44 + NN_PARAMS * 24), "flops": case["steps"] * case["batch"] * NN_TRAIN}
    if k == "infer":
        return {"bytes": case["samples"] * 44, "flops": case["samples"] * NN_FORWARD}
    if k == "batch":
        side = np.array([max(16, int(case["side"] * f)) for f in np.linspace(0.2, 1.0, case["scenes"])])
        tris = case["triangles"] * float(np.sum(np.linspace(0.1, 1.9, case["scenes"]) ** 2))
        return {"bytes": 9 * float(np.sum(side * side)) + 72 * tris, "flops": 84 * tris * 3}
    pixels = 9 * case["w"] * case["h"]
    if k == "objects":
        v = (case["rings"] + 1) * (case["segs"] + 1) if case["rings"] else 24
        n = 6 * case["rings"] * case["segs"] if case["rings"] else 36
        # each object's vertices and indices are read for its draw
        return {"bytes": pixels + case["objects"] * (20 * v + case["index"] * n) + 4 * case["texture"] ** 2,
                "flops": case["objects"] * v * 84}
    if k == "triangles":
        return {"bytes": pixels + 72 * case["n"], "flops": 28 * 3 * case["n"]}
    if k == "mix":
        return {"bytes": pixels + 32 * (3 * case["triangles"] + 2 * case["lines"] + case["points"]), "flops": 28 * 3 * case["triangles"]}
    geometry = 32 * (case["nx"] + 1) * (case["nz"] + 1) + 24 * case["nx"] * case["nz"]
    area = case["w"] * case["h"]
    if k == "capture":
        return {"bytes": 5 * (geometry + pixels) + 44 * case["keep"] * area, "flops": SHADE_TERRAIN * area}
    return {"bytes": case["views"] * (geometry + pixels),
            "flops": case["views"] * (NN_FORWARD if case["neural"] else SHADE_TERRAIN) * area}


# ------------------------------------------------------------------- exact

def forward64(p, x):
    """The network in 64 bits: output and what the backward pass needs."""
    W1, b1_, W2, b2, W3, b3 = p
    ang = 2 * math.pi * (torch.from_numpy(NN_STEPS).double() * x)[:, :, None] * torch.arange(1, 33, dtype=torch.float64)
    e = torch.stack([torch.sin(ang), torch.cos(ang)], -1).reshape(x.shape[0], 512)
    z1 = e @ W1.T + b1_
    h1 = z1.clamp(min=0)
    z2 = h1 @ W2.T + b2
    h2 = z2.clamp(min=0)
    return h2 @ W3.T + b3, (e, z1, h1, z2, h2)


def split(p):
    parts, at = [], 0
    for shape in ((64, 512), (64,), (64, 64), (64,), (3, 64), (3,)):
        n = math.prod(shape)
        parts.append(p[at:at + n].reshape(shape))
        at += n
    return parts


def batch_rows(step, batch, n):
    """The training sampler: a hash of (seed, step, slot) modulo the samples."""
    with np.errstate(over="ignore"):
        z = np.uint64(TRAIN_SEED) + np.uint64(0x9E3779B97F4A7C15) * (np.uint64(step * batch + 1) + np.arange(batch, dtype=np.uint64))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return ((z ^ (z >> np.uint64(31))) % np.uint64(n)).astype(np.int64)


def exact(case, seed):
    """Frames and captured samples have none: coverage, depth and colour are
    defined by the reference renderer's sequence of 32-bit operations."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "infer":
        p = [t for t in split(torch.from_numpy(net_params(rng)).double())]
        x = torch.from_numpy(samples(rng, case["samples"])[0]).double()
        return torch.cat([forward64(p, c)[0] for c in x.split(65536)])
    if case["kind"] == "train":
        flat = torch.from_numpy(net_params(rng)).double()
        x, t = (torch.from_numpy(v).double() for v in samples(rng, case["samples"]))
        m, v, losses, steps = torch.zeros_like(flat), torch.zeros_like(flat), [], case["steps"]
        for k in range(steps):
            rows = torch.from_numpy(batch_rows(k, case["batch"], case["samples"]))
            p = split(flat)
            y, (e, z1, h1, z2, h2) = forward64(p, x[rows])
            d = y - t[rows]
            losses.append(float((d * d).mean()))
            dy = 2 * d / d.numel()
            dz2 = (dy @ p[4]) * (z2 > 0)
            dz1 = (dz2 @ p[2]) * (z1 > 0)
            g = torch.cat([(dz1.T @ e).ravel(), dz1.sum(0), (dz2.T @ h1).ravel(), dz2.sum(0), (dy.T @ h2).ravel(), dy.sum(0)])
            lr = TRAIN_LR[1] + (TRAIN_LR[0] - TRAIN_LR[1]) * 0.5 * (1 + math.cos(math.pi * k / steps))
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            flat = flat - lr * (m / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1 - 0.999 ** (k + 1))) + 1e-8)
        return {"params": flat, "loss": torch.tensor(losses, dtype=torch.float64)}
    return None
