"""Frames and differentiable images of one context on several streams: the
context keeps its caller's stream, and its calls follow each other, so frames
that share its scratch memory equal those rendered alone.  Bar: equal bytes."""
import ctypes as C

import numpy as np
import pytest
import torch

from blackhole_8_amd import abi, diff, scenes
from blackhole_8_amd.render import Renderer

pytestmark = pytest.mark.gpu

SIZES = ((1920, 1080), (317, 179))


def _frame(r, k):
    w, h = SIZES[k % 2]
    p = scenes.disc_orbit(w, h, frames=8)
    p = p.with_camera(p.cameras[k % 8])
    rgb = torch.empty((h, w, 3), dtype=torch.uint8, device="cuda")
    hit = torch.empty((h, w), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()

    def launch():
        o = abi.Outputs(rgb.data_ptr(), hit.data_ptr())
        r._check(r.lib.bh_render_device(r.ctx, C.byref(p.scene), C.byref(p.options), C.byref(o)))

    return p, rgb, hit, launch


@pytest.fixture(scope="module")
def r():
    r = Renderer(0)
    r.set_textures(scenes.disc_orbit(8, 8).textures)
    yield r
    torch.cuda.synchronize()
    r.close()


@pytest.mark.parametrize("moves", [False, True])
def test_frames_between_images(r, moves):
    dr = diff.DiffRenderer(r, diff.DiffConfig(width=130, height=70))
    want = dr.forward(diff.FIT_START).cpu()
    st = [torch.cuda.Stream() for _ in range(2)]
    frames, images = [], []
    jobs = [_frame(r, k) for k in range(8)]
    for k, job in enumerate(jobs):
        print(f"[case] frame {k} and an image, stream {'moves' if moves else 'stays'}", flush=True)
        if k == 0 or moves:
            r._check(r.lib.bh_ctx_set_stream(r.ctx, C.c_void_p(st[k % 2].cuda_stream)))
        job[3]()
        images.append(dr.forward(diff.FIT_START))
    r._check(r.lib.bh_synchronize(r.ctx))
    torch.cuda.synchronize()
    r._check(r.lib.bh_ctx_set_stream(r.ctx, None))
    for k, (p, rgb, hit, _) in enumerate(jobs):
        solo = r.render(p.scene, p.options, ("rgb", "hit"))
        assert np.array_equal(rgb.cpu().numpy(), solo["rgb"]), k
        assert np.array_equal(hit.cpu().numpy(), solo["hit"]), k
        assert torch.equal(images[k].cpu(), want), k


def test_first_calls_of_a_context_in_a_capture():
    """A new context whose first image and gradient, and whose move to the
    capturing stream, come inside a capture; every replay equals the eager
    calls."""
    print("[case] first calls in a capture", flush=True)
    p = scenes.disc_orbit(317, 179)
    w, h = 130, 70
    weights = (torch.rand((h, w, 3), generator=torch.Generator().manual_seed(2)) + 0.5).cuda()
    frame = torch.zeros((179, 317, 3), dtype=torch.uint8, device="cuda")
    o = abi.Outputs(frame.data_ptr())
    graph = torch.cuda.CUDAGraph()
    with Renderer(0) as own:
        own.set_textures(p.textures)
        dr = diff.DiffRenderer(own, diff.DiffConfig(width=w, height=h))
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            rgb = dr.forward(diff.FIT_START)
            grad = dr.adjoint(diff.FIT_START, weights)
            own._check(own.lib.bh_ctx_set_stream(
                own.ctx, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
            own._check(own.lib.bh_render_device_noalloc(
                own.ctx, C.byref(p.scene), C.byref(p.options), C.byref(o)))
        own._check(own.lib.bh_ctx_set_stream(own.ctx, None))
        want = dr.forward(diff.FIT_START).cpu()
        want_grad = dr.adjoint(diff.FIT_START, weights).cpu()
        solo = own.render(p.scene, p.options, ("rgb",))["rgb"]
        for _ in range(3):
            rgb.zero_(), grad.zero_(), frame.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(rgb.cpu(), want) and torch.equal(grad.cpu(), want_grad)
            assert np.array_equal(frame.cpu().numpy(), solo)
            assert torch.equal(dr.forward(diff.FIT_START).cpu(), want)
        torch.cuda.synchronize()
