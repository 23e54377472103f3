"""The measured cases: what a user of this library has it do, through its
public entry points.

A case is one call of one kind:
  frame  one frame into the caller's device planes (bh_render_device)
  batch  many scenes of uneven size in one call (bh_render_batch_device)
  path   a camera path replayed from its graph and read back frame by frame
         (Renderer.path: launch, then read)
  diff   the differentiable render: the forward image, or the image and the
         gradient of a weighted sum of it in the four fitted parameters
         (DiffRenderer, diff.render)
  flat   one frame of the flat-space march (bh_render_flat_device)

Scenes (lengths in r_s unless said): `hole` the hole alone with an escape
background, camera at 15; `disc` the hole and its thin disc 3..12, camera at
20 and 80 deg, as on the 120-frame orbit; `shipped` the reference program's
own scene (mass 10, disc 100..1000, camera 2000 away); `spheres` the hole and
16 textured spheres with escape.  The seed picks what changes between two
calls of a program: the camera's place on its orbit, the disc's spin, the
spheres, the textures, the fit's parameters and weights.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

from blackhole_8_amd import abi, diff, scenes
from blackhole_8_amd.render import Renderer

DEV = "cuda:0"
PIXEL = {"rgb": 3, "hit": 1, "phi": 8, "hitpt": 24, "steps": 4}  # bytes a pixel
PLANES = {"rgb_hit": ("rgb", "hit"), "steps": ("rgb", "hit", "steps"),
          "all": ("rgb", "hit", "phi", "hitpt", "steps")}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _frame(scene, width, height, precision, planes="rgb_hit", nstep=20):
    return {"kind": "frame", "scene": scene, "width": width, "height": height,
            "precision": precision, "planes": planes, "nstep": nstep}


def listed():
    return [
        # the hole alone in FP64 with every plane: what a numerical study of
        # the lensing asks for (angles, hit points and step counts per pixel)
        dict(_frame("hole", 320, 180, "fp64", "all"), name="hole_320x180_fp64_planes"),
        # the demo program's own frame, in its default precision
        dict(_frame("shipped", 960, 540, "fp64"), name="shipped_960x540_fp64"),
        # a thumbnail: the smallest call, where the launches count
        dict(_frame("disc", 160, 90, "fp32"), name="disc_160x90_fp32"),
        # one frame of the 1080p orbit, the headline scene, on its own
        dict(_frame("disc", 1920, 1080, "fp32"), name="disc_1920x1080_fp32"),
        # an 8K still: the largest single frame
        dict(_frame("disc", 7680, 4320, "fp32"), name="disc_7680x4320_fp32"),
        # a scene with objects and a sky, at 720p
        dict(_frame("spheres", 1280, 720, "fp32"), name="spheres_1280x720_fp32"),
        # a data set: 512 uneven scenes, sides 32..1024, in one call
        {"kind": "batch", "count": 512, "side_lo": 32, "side_hi": 1024, "layout": 768,
         "name": "batch_512_uneven"},
        # a preview of a camera path, read back for the writer
        {"kind": "path", "frames": 24, "width": 480, "height": 270,
         "name": "path_24x480x270_read"},
        # the fit's target and its images: differentiable forward
        {"kind": "diff", "size": 512, "precision": "fp32", "grad": False,
         "name": "diff_forward_512_fp32"},
        # one iteration of the fit: image and gradient through autograd
        {"kind": "diff", "size": 512, "precision": "fp32", "grad": True,
         "name": "diff_gradient_512_fp32"},
        # the gradient in FP64, as a gradient check runs it
        {"kind": "diff", "size": 64, "precision": "fp64", "grad": True,
         "name": "diff_gradient_64_fp64"},
        # the flat-space program's frame at its own size
        {"kind": "flat", "width": 800, "height": 450, "steps": 10, "planes": "rgb_hit",
         "name": "flat_800x450"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("frame", "frame", "frame", "frame", "batch", "path", "diff", "diff",
                       "flat"))
    if kind == "frame":
        scene = rng.choice(("hole", "disc", "disc", "shipped", "spheres"))
        precision = rng.choice(("fp32", "fp32", "fp64"))
        big = {"fp32": 3840, "fp64": 1920}[precision] if scene in ("disc", "shipped") else 1280
        w = _log(rng, 96, big)
        h = max(32, int(w / rng.uniform(1.0, 2.0)))
        planes = rng.choice(("rgb_hit", "rgb_hit", "steps", "all"))
        nstep = rng.choice((20, 20, 20, rng.randint(10, 40)))
        if planes == "all" and w * h > 600000:
            planes = "steps"
        return _frame(scene, w, h, precision, planes, nstep)
    if kind == "batch":
        return {"kind": "batch", "count": _log(rng, 4, 512), "side_lo": 32,
                "side_hi": _log(rng, 128, 1024), "layout": rng.randint(1, 1 << 20)}
    if kind == "path":
        w = _log(rng, 160, 640)
        return {"kind": "path", "frames": rng.randint(2, 32), "width": w,
                "height": int(w * rng.uniform(0.5, 1.0))}
    if kind == "diff":
        precision = rng.choice(("fp32", "fp32", "fp64"))
        return {"kind": "diff", "size": _log(rng, 48, 768 if precision == "fp32" else 256),
                "precision": precision, "grad": rng.random() < 0.6}
    w = _log(rng, 160, 1920)
    return {"kind": "flat", "width": w, "height": max(32, int(w / rng.uniform(1.0, 2.0))),
            "steps": rng.randint(6, 20), "planes": rng.choice(("rgb_hit", "all"))}


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _unit(v):
    n = math.sqrt(sum(x * x for x in v))
    return [x / n for x in v]


def _cross(a, b):
    return [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]


def _look(position, width, height, fov):
    """Camera at position looking at the origin with +z up."""
    x = _unit([-p for p in position])
    k = x[2]
    z = _unit([-(0.0 - k * x[0]), -(0.0 - k * x[1]), -(1.0 - k * x[2])])
    return {"position": [float(p) for p in position], "x": x, "y": _unit(_cross(z, x)), "z": z,
            "width": width, "height": height, "fov": fov}


def _orbit(dist, incl, azim, width, height, fov):
    return _look([dist * math.sin(incl) * math.cos(azim), dist * math.sin(incl) * math.sin(azim),
                  dist * math.cos(incl)], width, height, fov)


def _square(half, spin=0.0):
    """The disc's texture square, corners p1..p4, turned about z."""
    c, s = math.cos(spin), math.sin(spin)
    return [[c * x - s * y, s * x + c * y, 0.0]
            for x, y in ((half, half), (-half, half), (-half, -half), (half, -half))]


def _scene_of(case, seed):
    """One frame's scene as plain numbers."""
    rng = random.Random(seed * 1000003 + 17)
    w, h = case["width"], case["height"]
    sc = {"mass": 0.5, "disc": None, "spheres": [], "background": False, "escape": False}
    kind = case["scene"]
    if kind == "disc":
        azim = math.radians(3.0 * rng.randrange(120) + rng.uniform(-1.0, 1.0))
        sc["cam"] = _orbit(20.0, math.radians(80.0), azim, w, h, math.pi / 3)
        sc["disc"] = {"p": _square(12.0), "r_out": 12.0, "r_in": 3.0}
    elif kind == "shipped":
        sc["cam"] = {"position": [-2000.0 + rng.uniform(-40, 40), rng.uniform(-40, 40), 400.0],
                     "x": [1.0, 0.0, 0.0], "y": [0.0, -1.0, 0.0], "z": [0.0, 0.0, -1.0],
                     "width": w, "height": h, "fov": math.pi / 2}
        sc["mass"] = 10.0
        p = _square(1000.0)
        p[2][1] = -64.0
        a = rng.uniform(0.0, 2.0 * math.pi)
        c, s = math.cos(a), math.sin(a)
        p = [[c * x - s * y, s * x + c * y, 0.0] for x, y, _ in p]
        sc["disc"] = {"p": p, "r_out": 1000.0, "r_in": 100.0}
    else:
        pos = [-15.0, rng.uniform(-0.5, 0.5), rng.uniform(-0.5, 0.5)]
        sc["cam"] = {"position": pos, "x": [1.0, 0.0, 0.0], "y": [0.0, -1.0, 0.0],
                     "z": [0.0, 0.0, -1.0], "width": w, "height": h, "fov": math.pi / 3}
        sc["background"] = sc["escape"] = True
        while kind == "spheres" and len(sc["spheres"]) < 16:
            rad = rng.uniform(0.3, 1.5)
            rr = rng.uniform(5.0 ** 3, 30.0 ** 3) ** (1.0 / 3.0)
            z, ph = rng.uniform(-1.0, 1.0), rng.uniform(0.0, 2.0 * math.pi)
            q = math.sqrt(max(0.0, 1.0 - z * z))
            c = [rr * q * math.cos(ph), rr * q * math.sin(ph), rr * z]
            if math.dist(c, pos) >= rad + 0.5:
                sc["spheres"].append((c, rad))
    return sc


def _disc_texture(seed, size=1024):
    """Radial bands with noise, as a photographed or painted disc has."""
    g = np.random.default_rng(seed)
    y, x = np.mgrid[0:size, 0:size]
    band = (np.hypot(x - size / 2, y - size / 2) / 32).astype(np.int64) % 2
    img = np.empty((size, size, 4), np.uint8)
    img[..., :3] = (64 + 128 * band)[..., None] + g.integers(0, 64, (size, size, 3))
    img[..., 3] = 255
    return img


def _sky(seed, rows=1024, cols=2048):
    g = np.random.default_rng(seed)
    y, x = np.mgrid[0:rows, 0:cols]
    check = (x * 16 // cols + y * 8 // rows) % 2
    return ((64 + 128 * check)[..., None] + g.integers(0, 64, (rows, cols, 3))).astype(np.uint8)


def _abi_camera(c):
    cam = abi.Camera()
    cam.position[:], cam.axis_x[:], cam.axis_y[:], cam.axis_z[:] = (c["position"], c["x"], c["y"],
                                                                   c["z"])
    cam.width, cam.height, cam.fov = c["width"], c["height"], c["fov"]
    return cam


def _abi_scene(sc):
    s = abi.Scene()
    s.camera = _abi_camera(sc["cam"])
    s.hole.mass = sc["mass"]
    s.background = scenes.SLOT_BG if sc["background"] else -1
    if sc["disc"]:
        d = sc["disc"]
        s.has_disc = 1
        s.disc = scenes.annulus(*d["p"], d["r_out"], d["r_in"], scenes.SLOT_DISC)
    for i, (c, rad) in enumerate(sc["spheres"]):
        s.spheres[i].center[:] = c
        s.spheres[i].radius = rad
        s.spheres[i].texture = scenes.SLOT_SPHERE0 + i
    s.n_spheres = len(sc["spheres"])
    return s


def _options(sc, precision, nstep):
    return scenes.options(precision=abi.PREC_FP64 if precision == "fp64" else abi.PREC_FP32,
                          nstep=nstep, escape=sc["escape"],
                          r_escape=100.0 if sc["escape"] else 0.0)


def _textures(r, sc, seed):
    if sc["background"]:
        r.set_texture(scenes.SLOT_BG, _sky(seed))
    if sc["disc"]:
        r.set_texture(scenes.SLOT_DISC, _disc_texture(seed + 1))
    g = np.random.default_rng(seed + 2)
    for i in range(len(sc["spheres"])):
        r.set_texture(scenes.SLOT_SPHERE0 + i, g.integers(0, 256, (256, 256, 3), np.uint8))


_stream = None


class State:
    """What a program keeps between calls; everything runs on one stream."""

    def __init__(self, case):
        global _stream
        if _stream is None:
            _stream = torch.cuda.Stream(DEV)
        self.case = case
        self.path = None
        self.r = Renderer(0)
        self.r._check(self.r.lib.bh_ctx_set_stream(self.r.ctx, C.c_void_p(_stream.cuda_stream)))

    def __del__(self):
        if self.path is not None:
            self.path.close()
        self.r.close()


def _planes(names, height, width):
    shape = {"rgb": ((height, width, 3), torch.uint8), "hit": ((height, width), torch.uint8),
             "phi": ((height, width), torch.float64), "hitpt": ((height, width, 3), torch.float64),
             "steps": ((height, width), torch.int32)}
    out = {k: torch.empty(shape[k][0], dtype=shape[k][1], device=DEV) for k in names}
    o = abi.Outputs(*[out[k].data_ptr() if k in out else None for k in PIXEL])
    return out, o


def _batch_sides(case):
    rng = random.Random(case["layout"])
    return [_log(rng, case["side_lo"], case["side_hi"]) for _ in range(case["count"])]


def prepare(case, seed):
    st = State(case)
    r, kind = st.r, case["kind"]
    if kind == "frame":
        sc = _scene_of(case, seed)
        _textures(r, sc, seed)
        st.scene, st.opts = _abi_scene(sc), _options(sc, case["precision"], case["nstep"])
        st.out, st.abi_out = _planes(PLANES[case["planes"]], case["height"], case["width"])
    elif kind == "batch":
        rng = random.Random(seed * 7919 + 3)
        sides = _batch_sides(case)
        px = [s * s for s in sides]
        n, total = len(sides), sum(px)
        r.set_texture(scenes.SLOT_DISC, _disc_texture(seed + 1))
        st.scenes, st.opts, st.outs = (abi.Scene * n)(), (abi.Options * n)(), (abi.Outputs * n)()
        st.out = {"rgb": torch.empty(total * 3, dtype=torch.uint8, device=DEV),
                  "hit": torch.empty(total, dtype=torch.uint8, device=DEV)}
        at = 0
        for i, side in enumerate(sides):
            rs = rng.uniform(0.5, 2.0)
            cam = _orbit(rng.uniform(6.0, 50.0) * rs,
                         math.radians(max(1e-3, rng.uniform(0.0, 90.0))),
                         rng.uniform(0.0, 2.0 * math.pi), side, side, math.pi / 3)
            disc = {"p": _square(12.0 * rs), "r_out": 12.0 * rs, "r_in": 3.0 * rs}
            sc = {"cam": cam, "mass": rs / 2.0, "disc": disc if rng.random() < 0.5 else None,
                  "spheres": [], "background": False, "escape": False}
            st.scenes[i], st.opts[i] = _abi_scene(sc), _options(sc, "fp32", 20)
            st.outs[i].rgb = st.out["rgb"].data_ptr() + 3 * at
            st.outs[i].hit = st.out["hit"].data_ptr() + at
            at += px[i]
    elif kind == "path":
        sc = _scene_of(dict(case, scene="disc"), seed)
        _textures(r, sc, seed)
        rng = random.Random(seed + 5)
        a0 = rng.uniform(0.0, 2.0 * math.pi)
        cams = [_abi_camera(_orbit(20.0, math.radians(80.0), a0 + math.radians(3.0 * k),
                                   case["width"], case["height"], math.pi / 3))
                for k in range(case["frames"])]
        st.path = r.path(_abi_scene(sc), _options(sc, "fp32", 20), cams)
    elif kind == "diff":
        r.set_texture(1, _disc_texture(seed + 1))
        prec = abi.PREC_FP64 if case["precision"] == "fp64" else abi.PREC_FP32
        st.dr = diff.DiffRenderer(r, diff.DiffConfig(width=case["size"], height=case["size"],
                                                     precision=prec))
        st.theta = torch.tensor(_theta(seed), dtype=torch.float64, requires_grad=case["grad"])
        st.weights = _weights(case, seed)
    else:
        st.scene, tex = _flat_scene(case, seed)
        r.set_textures(tex)
        st.out, st.abi_out = _planes(PLANES[case["planes"]], case["height"], case["width"])
    return st


def _theta(seed):
    rng = random.Random(seed * 31 + 7)
    return [t * rng.uniform(0.97, 1.03) for t in diff.FIT_TRUE]


def _weights(case, seed):
    g = torch.Generator(DEV).manual_seed(seed + 11)
    return torch.rand((case["size"], case["size"], 3), generator=g, device=DEV) + 0.5


def _flat_scene(case, seed):
    """The flat program's scene: three textured rectangles and the ground
    plane, the camera a little moved and turned, as its keys do."""
    s, tex = scenes.flat_test(case["width"], case["height"])
    rng = random.Random(seed + 23)
    s.camera.position[:] = [p + rng.uniform(-10.0, 10.0) for p in s.camera.position]
    s.steps = case["steps"]
    g = np.random.default_rng(seed)
    return s, {k: g.integers(0, 256, v.shape, np.uint8) for k, v in tex.items()}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    r, kind = st.r, st.case["kind"]
    if kind == "frame":
        r._check(r.lib.bh_render_device(r.ctx, C.byref(st.scene), C.byref(st.opts),
                                        C.byref(st.abi_out)))
        return st.out
    if kind == "batch":
        r._check(r.lib.bh_render_batch_device(r.ctx, len(st.scenes), st.scenes, st.opts, st.outs,
                                              None, None, None))
        return st.out
    if kind == "path":
        st.path.launch()
        frames = [st.path.read(k) for k in range(st.path.n)]
        return {"rgb": [f[0] for f in frames], "hit": [f[1] for f in frames]}
    if kind == "diff":
        if not st.case["grad"]:
            rgb, hit = st.dr.forward(st.theta.tolist(), with_hit=True)
            return {"rgb": rgb, "hit": hit}
        st.theta.grad = None
        img = diff.render(st.theta, st.dr)
        img.backward(st.weights)
        return {"rgb": img.detach(), "grad": st.theta.grad}
    r._check(r.lib.bh_render_flat_device(r.ctx, C.byref(st.scene), C.byref(st.abi_out)))
    return st.out


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every output plane once, and at most one texel a pixel (or the
    texture once, where that is less).  Operations: the reference's step rule
    in its reduced orbit-plane form (blackhole_8_amd/flops.py: 240 a ray, 35 a
    step with a disc, 30 without, 40 a hit) over the mean steps of the scene."""
    kind = case["kind"]
    if kind == "frame":
        px = case["width"] * case["height"]
        out = sum(PIXEL[k] for k in PLANES[case["planes"]])
        steps = {"disc": 25, "shipped": 30, "hole": 55, "spheres": 50}[case["scene"]]
        ops = 240 + (35 if case["scene"] in ("disc", "shipped") else 30) * steps \
            * case["nstep"] / 20 + 40
        if case["scene"] == "spheres":
            ops += 9 + 7 * 16 + 20 * steps
        tex = {"disc": 4 << 20, "shipped": 4 << 20, "hole": 8 << 20, "spheres": 12 << 20}
        return {"bytes": px * out + min(4 * px, tex[case["scene"]]), "flops": px * ops}
    if kind == "batch":
        px = sum(s * s for s in _batch_sides(case))
        return {"bytes": px * 4 + min(4 * px, 4 << 20), "flops": px * 1350.0}
    if kind == "path":
        px = case["width"] * case["height"] * case["frames"]
        return {"bytes": px * 4 + min(4 * px, 4 << 20), "flops": px * 1150.0}
    if kind == "diff":
        px = case["size"] ** 2
        return {"bytes": px * (24 if case["grad"] else 13) + min(16 * px, 4 << 20),
                "flops": px * (240 + 35 * 32) * (3.0 if case["grad"] else 1.0)}
    px = case["width"] * case["height"]
    out = sum(PIXEL[k] for k in PLANES[case["planes"]])
    return {"bytes": px * out + min(4 * px, 2 << 20), "flops": px * 40.0 * case["steps"]}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch
# ---------------------------------------------------------------------------
def _t(v):
    return torch.tensor(v, dtype=torch.float64, device=DEV)


def _dot(a, b):
    return (a * b).sum(-1)


def _segment(p1, p2, centre, radius):
    """Nearest entry of the segments p1..p2 into a sphere: (hit, point)."""
    a, b = p1 - centre, p2 - centre
    inside = (_dot(a, a).sqrt() < radius) & (_dot(b, b).sqrt() < radius)
    q = b - a
    qd, qq = _dot(q, a), _dot(q, q)
    cc = qd * qd - qq * (_dot(a, a) - radius * radius)
    t = (-qd - cc.clamp(min=0.0).sqrt()) / qq
    return ~inside & (cc > 0) & (t > 0) & (t < 1), a + q * t[:, None] + centre


def _annulus(p1, p2, n, r_in, r_out):
    t1, t2 = _dot(p1, n), _dot(p2, n)
    c = (p1 * t2.abs()[:, None] + p2 * t1.abs()[:, None]) / (t1.abs() + t2.abs())[:, None]
    rho = _dot(c, c).sqrt()
    return (t1 * t2 < 0) & (rho <= r_out) & (rho >= r_in), c


def _exact_frame(case, seed):
    """phi_end and the hit points of the reference's march: the 20-step
    bisection for the turning point, the trapezoid sum, straight chords."""
    sc = _scene_of(case, seed)
    cam, nstep, M = sc["cam"], case["nstep"], sc["mass"]
    W, H = case["width"], case["height"]
    N = W * H
    y, x = torch.meshgrid(torch.arange(H, device=DEV), torch.arange(W, device=DEV), indexing="ij")
    sx, sy = W / 2.0 - x.reshape(-1).double(), H / 2.0 - y.reshape(-1).double()
    f = W / (2.0 * math.tan(cam["fov"] / 2.0))
    pv = _t(cam["x"]) * f - _t(cam["y"]) * sx[:, None] - _t(cam["z"]) * sy[:, None]
    F = _t(cam["position"]).expand(N, 3)
    yv = F - pv
    yv = yv / _dot(yv, yv).sqrt()[:, None]
    zv = torch.linalg.cross(pv, yv)
    nz = _dot(zv, zv).sqrt()
    bad = ~(nz > 0)
    zv = zv / torch.where(bad, torch.ones_like(nz), nz)[:, None]
    xv = torch.linalg.cross(yv, zv)
    b, Y0, r0 = _dot(xv, F), _dot(yv, F), _dot(F, F).sqrt()
    ib2 = 1.0 / (b * b)
    lo = torch.full_like(b, math.ulp(1.0) ** (1.0 / 3.0))
    hi = torch.full_like(b, 1.0 / (3.0 * M))
    for _ in range(20):
        mid = (lo + hi) / 2.0
        up = mid * mid * (2.0 * M * mid - 1.0) + ib2 > 0
        lo, hi = torch.where(up, mid, lo), torch.where(up, hi, mid)
    captured = b < 3.0 * math.sqrt(3.0) * M
    u = 1.0 / r0
    du = (torch.where(captured, torch.full_like(b, 1.0 / (3.0 * M)), lo) - u) / nstep
    phi = torch.atan(b / Y0)
    w0 = torch.zeros_like(b)
    P = F.clone()
    live = ~bad
    point = torch.full((N, 3), math.nan, dtype=torch.float64, device=DEV)
    d = sc["disc"]
    if d:
        p = [_t(v) for v in d["p"]]
        n = torch.linalg.cross(p[2] - p[0], p[1] - p[0])
        n = n / _dot(n, n).sqrt()

    def meet(p1, p2, at):
        """The nearest object on the chords, for the rays `at`."""
        best = torch.full_like(b, math.inf)
        where = torch.zeros_like(p1)
        tests = [_segment(p1, p2, torch.zeros(3, dtype=torch.float64, device=DEV), 2.0 * M)]
        if d:
            tests.append(_annulus(p1, p2, n, d["r_in"], d["r_out"]))
        tests += [_segment(p1, p2, _t(c), rad) for c, rad in sc["spheres"]]
        for hit, q in tests:
            k = _dot(p1 - q, p1 - q)
            near = hit & at & (k < best)
            best = torch.where(near, k, best)
            where = torch.where(near[:, None], q, where)
        found = torch.isfinite(best)
        point[found] = where[found]
        return found

    def step(by, at):
        nonlocal u, phi, w0, P, live
        u = torch.where(at, u + du * by, u)
        w = 1.0 / (u * u * (2.0 * M * u - 1.0) + ib2).sqrt()
        phi = torch.where(at, phi + (w0 + w) * (du / 2.0), phi)
        w0 = torch.where(at, w, w0)
        r = (1.0 / u)[:, None]
        Q = yv * (r * phi.cos()[:, None]) + xv * (r * phi.sin()[:, None])
        live = live & ~meet(P, Q, at)
        P = torch.where(at[:, None], Q, P)

    for _ in range(nstep - 1):
        step(1.0, live)
    step(0.9, live)
    end = live & captured
    live = live & ~(meet(P, torch.zeros_like(P), end) | end)
    for _ in range(nstep - 1):
        step(-1.0, live)
    taken = 2 * nstep - 1
    while sc["escape"] and taken < 10000:
        on = live & ((u - du) * 100.0 > 1.0)
        if not bool(on.any()):
            break
        step(-1.0, on)
        taken += 1
    phi = torch.where(bad, torch.full_like(phi, math.nan), phi)
    return {"phi": phi.reshape(H, W), "hitpt": point.reshape(H, W, 3)}


def _exact_diff(case, seed):
    """The differentiable render with torch's own derivatives."""
    size, cfg = case["size"], diff.DiffConfig()
    tex = torch.from_numpy(_disc_texture(seed + 1)[..., :3].copy()).to(DEV).double()
    rows, cols = tex.shape[:2]
    theta = _t(_theta(seed)).requires_grad_(case["grad"])
    r_s, incl, dist, r_in = theta
    half, fw = cfg.r_outer, cfg.edge_width
    M = r_s / 2.0
    si, ci = torch.sin(incl), torch.cos(incl)
    F1 = torch.stack([dist * si * math.cos(cfg.azim), dist * si * math.sin(cfg.azim), dist * ci])
    ax = -F1 / _dot(F1, F1).sqrt()
    up = _t([0.0, 0.0, 1.0])
    az = -(up - ax * ax[2])
    az = az / _dot(az, az).sqrt()
    ay = torch.linalg.cross(az, ax)
    ay = ay / _dot(ay, ay).sqrt()
    g = torch.arange(size, device=DEV, dtype=torch.float64)
    sx = (size / 2.0 - g)[None, :].expand(size, size).reshape(-1, 1)
    sy = (size / 2.0 - g)[:, None].expand(size, size).reshape(-1, 1)
    f = size / (2.0 * math.tan(cfg.fov / 2.0))
    pv = ax * f - ay * sx - az * sy
    F = F1.expand_as(pv)
    yv = F - pv
    yv = yv / _dot(yv, yv).sqrt()[:, None]
    zv = torch.linalg.cross(pv, yv)
    cc = _dot(zv, zv)
    bad = ~(cc > 0)
    zv = zv / torch.where(bad, torch.ones_like(cc), cc).sqrt()[:, None]
    xv = torch.linalg.cross(yv, zv)
    b, Y0, r0 = _dot(xv, F), _dot(yv, F), _dot(F1, F1).sqrt()
    bad = bad | ~(b > 1e-9)  # through the centre: black, and no derivative
    b = torch.where(bad, torch.ones_like(b), b)
    xv = torch.where(bad[:, None], torch.zeros_like(xv), xv)
    e1, e2 = F / r0, (xv * Y0[:, None] - yv * b[:, None]) / r0
    ib2 = 1.0 / (b * b)
    captured = b < 3.0 * math.sqrt(3.0) * M
    with torch.no_grad():
        q = (27.0 * M * M * ib2).clamp(max=1.0)
        l = (0.5 + torch.sin(torch.asin(2.0 * q - 1.0) / 3.0)) / (3.0 * M)
        for _ in range(3):
            gp = l * (6.0 * M * l - 2.0)
            l = torch.where(gp < -1e-12, l - (l * l * (2.0 * M * l - 1.0) + ib2) / gp, l)
        gp = l * (6.0 * M * l - 2.0)
        gp = torch.where(gp < -1e-12, gp, torch.full_like(gp, -1e300))
    l = torch.where(captured, 1.0 / (3.0 * M), l - (l * l * (2.0 * M * l - 1.0) + ib2) / gp)
    n = 20
    u0 = 1.0 / r0
    du = (l - u0) / n
    R2 = (r_s * r_s).detach()
    one = torch.ones_like(b)
    T, psi, wp, P1 = one.clone(), torch.zeros_like(b), torch.zeros_like(b), F
    rgb = torch.zeros_like(pv)
    cls_alive = ~bad

    def smooth(v):
        t = (v + 0.5).clamp(0.0, 1.0)
        return t * t * (3.0 - 2.0 * t)

    for j in range(1, 2 * n):
        if j == n + 1:
            cls_alive = cls_alive & ~captured
        kj = float(j) if j < n else 2 * n - j - 0.1
        u = u0 + kj * du
        G = u * u * (2.0 * M * u - 1.0) + ib2
        w = 1.0 / torch.where(G > 0, G, one).sqrt()
        psi = psi + (wp + w) * (du / 2.0)
        wp = w
        P2 = (torch.cos(psi)[:, None] * e1 + torch.sin(psi)[:, None] * e2) / u[:, None]
        with torch.no_grad():
            d1, d2, Q = _dot(P1, P1), _dot(P2, P2), P2 - P1
            qd, qq = _dot(Q, P1), _dot(Q, Q)
            disc = qd * qd - qq * (d1 - R2)
            t = (-qd - disc.clamp(min=0.0).sqrt()) / qq
            hh = ~((d1 < R2) & (d2 < R2)) & (disc > 0) & (t > 0) & (t < 1)
            dh = t * t * qq
        z1, z2 = P1[:, 2], P2[:, 2]
        cross = (z1 * z2 < 0) & cls_alive
        sf = torch.where(cross, z1, 0.5 * one) / torch.where(cross, z1 - z2, one)
        c = P1 + sf[:, None] * (P2 - P1)
        rho = torch.where(cross, _dot(c, c), one).sqrt()
        al = smooth((rho - r_in) / fw) * smooth((half - rho) / fw)
        use = cross & (al > 0) & (~hh | (sf * sf * qq < dh))
        U = (half - c[:, 0]) * (cols / (2.0 * half)) - 0.5
        vv = (c[:, 1] - half) ** 2 + c[:, 2] ** 2
        V = torch.where(use, vv, one).sqrt() * (rows / (2.0 * half)) - 0.5
        fx, fy = U.detach().floor(), V.detach().floor()
        tx, ty = (U - fx)[:, None], (V - fy)[:, None]
        ix, iy = fx.clamp(-1, cols).long(), fy.clamp(-1, rows).long()
        x0, x1 = ix.clamp(0, cols - 1), (ix + 1).clamp(0, cols - 1)
        y0, y1 = iy.clamp(0, rows - 1), (iy + 1).clamp(0, rows - 1)
        top = tex[y0, x0] + (tex[y0, x1] - tex[y0, x0]) * tx
        bot = tex[y1, x0] + (tex[y1, x1] - tex[y1, x0]) * tx
        a = torch.where(use, al, torch.zeros_like(al))
        rgb = rgb + torch.where(use[:, None], (T * a)[:, None] * (top + (bot - top) * ty),
                                torch.zeros_like(rgb))
        T = T * (1.0 - a)
        cls_alive = cls_alive & ~hh & (T > 0)
        P1 = P2
    out = {"rgb": rgb.detach().reshape(size, size, 3)}
    if case["grad"]:
        wt = _weights(case, seed).double().reshape(-1, 3)
        out["grad"] = torch.autograd.grad((rgb * wt).sum(), theta)[0].cpu()
    return out


def _exact_flat(case, seed):
    """Hit points of the straight chords: camera to pixel point, then that
    vector again and again (lengthened to 100/|v|^2 of itself when short)."""
    s, _ = _flat_scene(case, seed)
    W, H = case["width"], case["height"]
    y, x = torch.meshgrid(torch.arange(H, device=DEV), torch.arange(W, device=DEV), indexing="ij")
    sx, sy = W / 2.0 - x.reshape(-1, 1).double(), H / 2.0 - y.reshape(-1, 1).double()
    cam = s.camera
    f = W / (2.0 * math.tan(cam.fov / 2.0))
    P1 = _t(cam.position[:]).expand(W * H, 3)
    P2 = _t(cam.axis_x[:]) * f - _t(cam.axis_y[:]) * sx - _t(cam.axis_z[:]) * sy
    v = P2 - P1
    d2 = _dot(v, v)[:, None]
    v = torch.where(d2 < 100.0, v * (100.0 / d2), v)
    live = torch.ones(W * H, dtype=torch.bool, device=DEV)
    point = torch.full((W * H, 3), math.nan, dtype=torch.float64, device=DEV)
    for _ in range(case["steps"]):
        best = torch.full((W * H,), math.inf, dtype=torch.float64, device=DEV)
        for i in range(s.n_rects + s.n_planes):
            if i < s.n_rects:
                a, b, d = (_t(s.rects[i].vertex[k][:]) for k in (1, 2, 4))
                n = torch.linalg.cross(b - a, d - a)
                n = n / _dot(n, n).sqrt()
            else:
                a, n = _t(s.planes[i - s.n_rects].position[:]), _t(s.planes[i - s.n_rects].axis_z[:])
            t1, t2 = _dot(P1 - a, n), _dot(P2 - a, n)
            q = ((P1 - a) * t2.abs()[:, None] + (P2 - a) * t1.abs()[:, None]) \
                / (t1.abs() + t2.abs())[:, None]
            hit = t1 * t2 < 0 if i < s.n_rects else t1 * t2 <= 0
            for e in ((b - a, d - a) if i < s.n_rects else ()):
                hit = hit & (_dot(q, e) > 0) & (_dot(q, e) < _dot(e, e))
            q = q + a
            k = _dot(P1 - q, P1 - q)
            near = hit & live & (k < best)
            best = torch.where(near, k, best)
            point = torch.where(near[:, None], q, point)
        live = live & ~torch.isfinite(best)
        P1, P2 = P2, P2 + v
    return {"phi": None, "hitpt": point.reshape(H, W, 3)}


def exact(case, seed):
    """phi_end and hit points of a frame with every plane, the differentiable
    image and gradient; bytes and whole numbers have no such value."""
    if case["kind"] == "flat" and case["planes"] == "all":
        return _exact_flat(case, seed)
    if case["kind"] == "frame" and case["planes"] == "all":
        return _exact_frame(case, seed)
    if case["kind"] == "diff":
        return _exact_diff(case, seed)
    return None
