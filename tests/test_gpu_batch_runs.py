"""Batches large enough that a wave of the grid mode marches a run of two to
four tiles, whose runs cross from one scene to the next: every scene equals its
solo render byte for byte, with its finish time within the call's."""
import pytest

from blackhole_8_amd import abi, scenes

import numpy as np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,side", [(18, 997), (37, 1003)])
def test_runs_of_tiles_equal_solo_renders(renderer, n, side):
    items = []
    for k in range(n):
        w, h = side - 8 * (k % 3), side + k % 5
        p = scenes.disc_orbit(w, h)
        s = abi.Scene.from_buffer_copy(p.scene)
        s.camera = scenes.orbit_camera(6.0 + 1.3 * k, 20.0 + 4.0 * k % 150, 31.0 * k, w, h, 1.0)
        s.has_disc = k % 3 != 1
        items.append((s, scenes.options(precision=abi.PREC_FP32)))
    renderer.set_textures(scenes.disc_orbit(8, 8).textures)
    print(f"[case] batch of {n} scenes of about {side}x{side}", flush=True)
    res = renderer.render_batch(items)
    timed, ms, st = renderer.render_batch(items, timing=True)
    assert (ms > 0).all() and (ms <= st.total_ms + 1e-3).all()
    for i, ((s, o), r, t) in enumerate(zip(items, res, timed)):
        solo = renderer.render(s, o, ("rgb", "hit"))
        for k in ("rgb", "hit"):
            assert np.array_equal(r[k], solo[k]), f"scene {i} {k}"
            assert np.array_equal(t[k], solo[k]), f"scene {i} {k} (timed)"
