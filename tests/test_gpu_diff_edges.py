"""Differentiable render at frames that are no multiple of its 16x16 tiles and
where lanes of a wave end at different steps, and a scene with a disc crossing
at the very end of its chord, whose recorded angle rounds to the other side.

Bars: the forward tests' own (classes identical but for 1e-4 of the pixels,
colour within 1/255 where they agree; FP64: identical, 1e-4); gradients of
FP32 against FP64 within 2e-2 of their norm (the FP32 image crosses texel cells
that the FP64 one does not, a few in a thousand)."""
import os

import numpy as np
import pytest
import torch

from blackhole_8_amd import abi, diff
from blackhole_8_amd.render import Renderer
import oracle

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module")
def dctx():
    r = Renderer(0)
    tex = diff.load_target_textures(r)
    yield r, tex
    r.close()


@pytest.mark.parametrize("w,h", [(1, 1), (17, 5), (63, 33), (130, 47)])
@pytest.mark.parametrize("prec", [abi.PREC_FP32, abi.PREC_FP64])
def test_forward_at_ragged_sizes(dctx, w, h, prec):
    print(f"[case] diff forward {w}x{h} prec {prec}", flush=True)
    dr = diff.DiffRenderer(dctx[0], diff.DiffConfig(width=w, height=h, precision=prec))
    rgb, hit = dr.forward(diff.FIT_START, with_hit=True)
    g = dr.adjoint(diff.FIT_START, torch.ones((h, w, 3)), want_rgb=True)
    torch.cuda.synchronize()
    assert torch.equal(g[1], rgb) and torch.isfinite(g[0]).all()
    rgb, hit = rgb.cpu().numpy().astype(np.float64), hit.cpu().numpy()
    orgb, ohit, _ = oracle.render_diff(dr.cfg.params(diff.FIT_START), dctx[1], THREADS)
    d = np.abs(rgb - orgb).max(axis=2)
    if prec == abi.PREC_FP64:
        assert (hit == ohit).all() and d.max() <= 1e-4
    else:
        assert (hit != ohit).sum() <= max(1, 1e-4 * w * h)
        assert (d[hit == ohit] <= 1.0).all()


def test_adjoint_where_a_crossing_ends_its_chord(dctx):
    theta = (1.2882127466191091, 1.2014177119371683, 18.930757082033107, 3.542348908958477)
    print("[case] diff adjoint, crossing at a chord's end, 512x512", flush=True)
    w = torch.rand((512, 512, 3), generator=torch.Generator().manual_seed(1)) + 0.5
    g = {}
    for prec in (abi.PREC_FP32, abi.PREC_FP64):
        dr = diff.DiffRenderer(dctx[0], diff.DiffConfig(precision=prec))
        g[prec] = dr.adjoint(theta, w).cpu()
        assert dr.overflow() == 0
    assert torch.isfinite(g[abi.PREC_FP32]).all()
    assert (g[abi.PREC_FP32] - g[abi.PREC_FP64]).norm() <= 2e-2 * g[abi.PREC_FP64].norm()
