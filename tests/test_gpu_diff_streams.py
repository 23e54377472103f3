"""The differentiable render on the streams of its callers: the null stream, a
stream of torch's and a captured graph give the bits of the calls on the
context's own stream, and a workspace that is too small is refused.  Bar:
equal bits, since the kernels and their reduction order are the same."""
import ctypes as C

import pytest
import torch

from blackhole_8_amd import abi, diff
from blackhole_8_amd.render import Renderer

pytestmark = pytest.mark.gpu

W, H = 70, 50


@pytest.fixture(scope="module")
def dr():
    r = Renderer(0)
    diff.load_target_textures(r)
    yield diff.DiffRenderer(r, diff.DiffConfig(width=W, height=H))
    torch.cuda.synchronize()
    r.close()


def weights():
    return torch.rand((H, W, 3), generator=torch.Generator().manual_seed(4)).cuda() + 0.5


@pytest.fixture(scope="module")
def own(dr):
    """The image and the gradient from the calls on the context's stream."""
    p, w = dr.cfg.params(diff.FIT_START), weights()
    rgb = torch.empty((H, W, 3), device="cuda")
    grad = torch.empty(4, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    r = dr.r
    r._check(r.lib.bh_diff_render_device(r.ctx, C.byref(p), dr.cfg.precision, rgb.data_ptr(), None))
    r._check(r.lib.bh_diff_adjoint_device(r.ctx, C.byref(p), dr.cfg.precision, w.data_ptr(), None,
                                          None, grad.data_ptr(), None))
    r._check(r.lib.bh_synchronize(r.ctx))
    return rgb.cpu(), grad.cpu()


@pytest.mark.parametrize("side", [False, True])
def test_current_stream(dr, own, side):
    print(f"[case] diff on {'a side' if side else 'the null'} stream {W}x{H}", flush=True)
    st = torch.cuda.Stream() if side else torch.cuda.default_stream()
    w = weights()
    st.wait_stream(torch.cuda.default_stream())
    with torch.cuda.stream(st):
        for _ in range(3):
            rgb = dr.forward(diff.FIT_START)
            grad, rgb2 = dr.adjoint(diff.FIT_START, w, want_rgb=True)
            a, b, c = rgb.cpu(), rgb2.cpu(), grad.cpu()
            assert torch.equal(a, own[0]) and torch.equal(b, own[0]) and torch.equal(c, own[1])
            assert dr.overflow() == 0


def test_captured(dr, own):
    print(f"[case] diff captured {W}x{H}", flush=True)
    w = weights()
    dr.adjoint(diff.FIT_START, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rgb = dr.forward(diff.FIT_START)
        grad = dr.adjoint(diff.FIT_START, w)
    for _ in range(3):
        rgb.zero_()
        grad.zero_()
        graph.replay()
        assert torch.equal(rgb.cpu(), own[0]) and torch.equal(grad.cpu(), own[1])
        assert torch.equal(dr.forward(diff.FIT_START).cpu(), own[0])
        torch.cuda.synchronize()


def test_small_workspace_is_refused(dr):
    r, p = dr.r, dr.cfg.params(diff.FIT_START)
    n = r.lib.bh_diff_work_bytes(W, H)
    assert n == 8 * 5 * ((W + 15) // 16) * ((H + 15) // 16)
    assert r.lib.bh_diff_work_bytes(0, H) == 0
    w, grad = weights(), torch.empty(4, dtype=torch.float64, device="cuda")
    work = torch.empty(n + 8, dtype=torch.uint8, device="cuda")
    for ptr, size in ((None, n), (work.data_ptr(), n - 1), (work.data_ptr() + 4, n)):
        rc = r.lib.bh_diff_adjoint_stream(r.ctx, None, C.byref(p), dr.cfg.precision, w.data_ptr(),
                                          None, None, grad.data_ptr(), None, ptr, size)
        assert rc == abi.BH_ERR_INVALID_ARG
