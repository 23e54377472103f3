"""The flat march places only the chords that can cross an object; the oracle
tests every chord against every object.  Random scenes over the forms a flat
scene takes: no objects, all slots, lengths from 1e-6 to 1e6, rectangles
without area, planes with a zero axis or through the camera, views along a
plane, from one chord to a thousand.  Bars: classes and step counts identical;
hit points within 1e-12 of the scene's size (both use the same operations in
the same order; the crossing's division may be rounded differently)."""
import math

import numpy as np
import pytest

from blackhole_8_amd import abi, scenes
import oracle

pytestmark = pytest.mark.gpu

ALL = ("rgb", "hit", "hitpt", "steps")


def _scene(rng, w, h, steps, scale):
    s, tex = scenes.flat_test(w, h)
    u = lambda k=3: rng.uniform(-300, 300, k) * scale
    pos = u()
    if rng.random() < 0.3:
        pos = np.zeros(3)
    cam = scenes.look_at(w, h, rng.uniform(0.2, 2.6), tuple(pos), tuple(u()))
    s.camera = cam
    s.steps = steps
    slot = s.rects[0].texture
    s.n_rects = int(rng.integers(0, abi_rects() + 1))
    spread = math.exp(rng.uniform(0.0, math.log(60.0)))  # the objects' distances in chords
    far = lambda: u() * spread
    for i in range(s.n_rects):
        p1, a, b = far(), far() * 0.5, far() * 0.5
        kind = rng.random()
        if kind < 0.1:
            a = b * 2.0           # no area
        elif kind < 0.4:
            p1[2] = a[2] = b[2] = 0.0
        for k, v in enumerate((p1, p1 + a, p1 + a + b, p1 + b)):
            s.rects[i].vertex[k + 1][:] = tuple(v)
        s.rects[i].texture = slot
    s.n_planes = int(rng.integers(0, abi_planes() + 1)) if rng.random() < 0.4 else 0
    for i in range(s.n_planes):
        pl = s.planes[i]
        kind = rng.random()
        pl.position[:] = tuple(pos) if kind < 0.1 else tuple(far())
        z = rng.normal(size=3)
        if kind < 0.2:
            z = np.zeros(3)
        elif kind < 0.5:          # the view's axis lies in the plane
            z = np.cross(np.array(cam.axis_x[:]), z)
        x = np.array([1.0, 0.1, 0.0])
        pl.axis_x[:], pl.axis_y[:], pl.axis_z[:] = tuple(x), (0.0, 1.0, 0.0), tuple(z)
        pl.pattern_size = 0.0 if rng.random() < 0.3 else float(rng.integers(1, 50))
    return s, tex


def abi_rects():
    return len(abi.FlatScene().rects)


def abi_planes():
    return len(abi.FlatScene().planes)


@pytest.mark.parametrize("steps", [1, 2, 7, 60, 1000])
@pytest.mark.parametrize("scale", [1e-6, 1.0, 1e6])
def test_random_scenes_match_the_oracle(renderer, steps, scale):
    rng = np.random.default_rng(int(steps * 7 + math.log10(scale)) & 0xffff)
    for k in range(12):
        w, h = int(rng.integers(1, 70)), int(rng.integers(1, 40))
        s, tex = _scene(rng, w, h, steps, scale)
        renderer.set_textures(tex)
        print(f"[case] flat {w}x{h} steps {steps} scale {scale} no {k}: "
              f"{s.n_rects} rects {s.n_planes} planes", flush=True)
        g, r = renderer.render_flat(s, ALL), oracle.render_flat(s, tex, ALL)
        assert np.array_equal(g["hit"], r["hit"])
        assert np.array_equal(g["steps"], r["steps"])
        assert np.array_equal(np.isnan(g["hitpt"]), np.isnan(r["hitpt"]))
        ok = ~np.isnan(r["hitpt"])
        size = 1e3 * max(scale, 1.0) + np.abs(r["hitpt"][ok]).max(initial=0.0)
        assert (np.abs(g["hitpt"][ok] - r["hitpt"][ok]) <= 1e-12 * size).all()
