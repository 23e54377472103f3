"""bh_steps_taken: the steps that the march takes of a ray that may end early
are no more than those of the reference's rule, the same where the ray ends at
an object, and none where the set-up ends it or leaves it to the FP64 pass.
Counts are whole numbers: equality."""
import numpy as np
import pytest

from blackhole_8_amd import abi, scenes
from blackhole_8_amd.render import BHError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nstep", [5, 20, 23])
@pytest.mark.parametrize("disc", [True, False])
def test_steps_taken_against_the_steps_plane(renderer, nstep, disc):
    p = scenes.disc_orbit(317, 179)
    s = abi.Scene.from_buffer_copy(p.scene)
    s.has_disc = int(disc)
    o = scenes.options(precision=abi.PREC_FP32, nstep=nstep)
    renderer.set_textures(p.textures)
    print(f"[case] steps taken nstep {nstep} disc {disc}", flush=True)
    out = renderer.render(s, o, ("hit", "steps"))
    taken = renderer.steps_taken(s, o)
    marched = taken > 0
    assert (taken <= out["steps"]).all() and (taken >= 0).all()
    if disc:
        at_disc = marched & (out["hit"] == abi.HIT_DISC)
        assert at_disc.sum() > 1000
        assert np.array_equal(taken[at_disc], out["steps"][at_disc])
        missed = marched & (out["hit"] == abi.HIT_NONE)
        assert (taken[missed] >= nstep).all()
        assert taken.sum() < out["steps"].sum()
    else:  # a hole alone: rays away from the band end in their set-up
        assert marched.mean() < 0.2


def test_frames_in_which_no_ray_ends_early_are_refused(renderer):
    for p in (scenes.spheres(64, 48), scenes.plain_hole(64, 48)):
        renderer.set_textures(p.textures)
        with pytest.raises(BHError):
            renderer.steps_taken(p.scene, p.options)
