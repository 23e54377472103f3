"""DiffRenderer.overflow() reports the last adjoint's count although adjoints
on several streams may end in any order: the host code on a stand-in for the
library and for torch's streams, which runs the launches in an order of the
test's."""
import ctypes as C

import pytest
import torch

from blackhole_8_amd import diff


class Stream:
    def __init__(self, handle):
        self.cuda_stream = handle
        self.waited = []

    def wait_stream(self, other):
        self.waited.append(other)


class Lib:
    """Keeps each adjoint's overflow word; finish() lets one end."""

    def __init__(self):
        self.calls = []

    def bh_ctx_set_stream(self, ctx, stream):
        return 0

    def bh_diff_work_bytes(self, w, h):
        return 64

    def bh_diff_adjoint_stream(self, ctx, stream, p, prec, g, rgb, hit, grad, ovf, work, n):
        self.calls.append(ovf)
        return 0

    def finish(self, call, count):
        C.c_uint32.from_address(self.calls[call]).value = count


class Context:
    ctx = None

    def __init__(self, lib):
        self.lib = lib

    def _check(self, rc):
        assert rc == 0


@pytest.mark.parametrize("order", [(0, 1), (1, 0)])
def test_overflow_is_the_last_adjoints(monkeypatch, order):
    current = [Stream(0)]
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: current[0])
    monkeypatch.setattr(torch.cuda, "Stream", lambda dev=None: Stream(99))
    monkeypatch.setattr(torch, "device", lambda *a: "cpu")
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, s: None)
    # (an earlier call's word stays writable here; on the GPU its memory is used
    # again only after that call on its stream)
    kept, empty = [], torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: kept.append(empty(*a, **k)) or kept[-1])
    lib = Lib()
    dr = diff.DiffRenderer(Context(lib), diff.DiffConfig(width=4, height=2))
    assert dr.overflow() == 0
    weights, counts, streams = torch.ones((2, 4, 3)), (7, 3), (Stream(1), Stream(2))
    for s in streams:
        current[0] = s
        dr.adjoint(diff.FIT_START, weights)
    for k in order:
        lib.finish(k, counts[k])
    current[0] = Stream(3)
    assert dr.overflow() == counts[1]
    assert current[0].waited == [streams[1]]
    current[0] = streams[1]
    assert dr.overflow() == counts[1] and streams[1].waited == []
