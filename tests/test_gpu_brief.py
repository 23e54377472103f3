"""Frames without the swept-angle plane end rays early (the march's brief form,
and rays whose class their set-up already tells): every other plane must be
byte for byte that of the frame with the swept angle, which marches each ray
to its end.  Scenes: no disc, discs seen from outside, inside and through,
cameras that look past or away from the hole, tilted discs, step counts on
both sides of the early ends' least one."""
import math

import numpy as np
import pytest

from blackhole_8_amd import abi, scenes

pytestmark = pytest.mark.gpu

W, H = 173, 101


def _disc(rng, r_out, r_in):
    n = np.array([rng.uniform(-1, 1), rng.uniform(-1, 1), rng.uniform(0.2, 1)])
    n /= np.linalg.norm(n)
    a = np.cross(n, [1.0, 0.0, 0.0])
    a /= np.linalg.norm(a)
    b = np.cross(n, a)
    k = r_out / math.sqrt(0.5)
    return scenes.annulus(a * k, b * k, -a * k, -b * k, r_out, r_in, scenes.SLOT_DISC)


def _scene(rng, dist, disc, aim):
    cam = scenes.orbit_camera(dist, rng.uniform(1, 179), rng.uniform(0, 360), W, H,
                              rng.uniform(0.3, 2.2), target=aim)
    p = scenes.disc_orbit(W, H)
    s = abi.Scene.from_buffer_copy(p.scene)
    # the camera's place is set from the hole; only its aim moves
    pos = scenes.orbit_camera(dist, 70.0, rng.uniform(0, 360), W, H, 1.0).position
    s.camera = scenes.look_at(W, H, cam.fov, tuple(pos), aim)
    s.has_disc = int(disc is not None)
    if disc is not None:
        s.disc = _disc(rng, *disc)
    return s


@pytest.mark.parametrize("nstep", [2, 4, 5, 9, 20, 37])
@pytest.mark.parametrize("disc", [None, (12.0, 3.0), (2.2, 0.4), (30.0, 0.0), (4.0, 3.9)])
def test_brief_planes_equal_the_full_march(renderer, nstep, disc):
    rng = np.random.default_rng(1000 * nstep + (0 if disc is None else int(10 * disc[0])))
    renderer.set_textures(scenes.disc_orbit(W, H).textures)
    for dist, aim in ((1.6, (0, 0, 0)), (6.5, (0, 0, 0)), (14.0, (3.0, -2.0, 1.0)),
                      (20.0, (60.0, 5.0, 0.0)), (48.0, (0, 0, 0))):
        s = _scene(rng, dist, disc, tuple(float(v) for v in aim))
        o = scenes.options(precision=abi.PREC_FP32, nstep=nstep)
        print(f"[case] brief march nstep {nstep} disc {disc} from {dist}", flush=True)
        full = renderer.render(s, o, ("rgb", "hit", "steps", "hitpt", "phi"))
        for want in (("rgb", "hit", "steps", "hitpt"), ("rgb", "hit")):
            got = renderer.render(s, o, want)
            for k in want:
                assert got[k].tobytes() == full[k].tobytes(), (k, dist)


@pytest.mark.parametrize("scale", [1e-3, 1e4, 1e6])
@pytest.mark.parametrize("disc", [None, (12.0, 3.0)])
def test_brief_planes_at_other_scales(renderer, scale, disc):
    """Lengths at which the turning point leaves its solver's bracket too."""
    rng = np.random.default_rng(7)
    renderer.set_textures(scenes.disc_orbit(W, H).textures)
    for dist in (6.5, 20.0, 48.0):
        s = _scene(rng, dist * scale, None if disc is None else (disc[0] * scale, disc[1] * scale),
                   (0.0, 0.0, 0.0))
        s.hole.mass *= scale
        o = scenes.options(precision=abi.PREC_FP32)
        print(f"[case] brief march at scale {scale} disc {disc} from {dist}", flush=True)
        full = renderer.render(s, o, ("rgb", "hit", "steps", "hitpt", "phi"))
        for want in (("rgb", "hit", "steps", "hitpt"), ("rgb", "hit")):
            got = renderer.render(s, o, want)
            for k in want:
                assert got[k].tobytes() == full[k].tobytes(), (k, dist)
