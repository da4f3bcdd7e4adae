"""The pinned words a kernel answers into (``_lib.HostWords``) are given back
only when nothing queued can write to them any more, also where a call
between queueing the write and reading it raises."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from ssla_amd import _lib, gla, scatter


@pytest.fixture
def log(monkeypatch):
    """HostWords without a device; what it does, in order."""
    seen = []

    class Pool(list):
        def append(self, w):
            assert not getattr(w, "pending", False)
            seen.append("back")
            super().append(w)

    def init(self, dev):
        own = dict(words=np.zeros(2, np.int64), dev=dev, ptr=0, handle=0, pending=False,
                   event=SimpleNamespace(synchronize=lambda: seen.append("event")))
        for nm in type(self).__slots__:
            setattr(self, nm, own[nm])

    def call(ret):
        def fn(*_):
            seen.append("queued")
            return ret
        return fn
    monkeypatch.setattr(_lib.HostWords, "__init__", init)
    monkeypatch.setattr(_lib.HostWords, "_free", {-1: Pool()})
    monkeypatch.setattr(_lib.HostWords, "_lost", [], raising=False)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *_: seen.append("device"))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    err = SimpleNamespace(ssla_seq_bounds_async=call(0), ssla_scatter_max_checked=call(_lib.SSLA_ERR_LAUNCH),
                          ssla_scatter_workspace_size=lambda *_: 16, ssla_last_error=lambda: b"launch")
    monkeypatch.setattr(_lib, "load", lambda: err)
    return seen


def _recurrent(monkeypatch, raises):
    x = torch.zeros(3, 1, 16)
    cu = torch.tensor([0, 3])
    monkeypatch.setattr(gla, "_prep", lambda *_: (x, x, x, x, cu, None))

    def rec(*a):
        if raises:
            raise raises
        return a[7], a[8]
    monkeypatch.setattr(gla, "_recurrent", rec)
    return lambda: gla.fused_recurrent_gla(x, x, x, x, SimpleNamespace(is_cuda=True))


def test_read_gives_back(log, monkeypatch):
    _recurrent(monkeypatch, None)()
    assert log == ["queued", "event", "back"]


@pytest.mark.parametrize("exc", [torch.OutOfMemoryError("no memory"), NotImplementedError(), KeyboardInterrupt()])
def test_recurrence_raises_after_the_bounds(log, monkeypatch, exc):
    with pytest.raises(type(exc)):
        _recurrent(monkeypatch, exc)()
    assert log == ["queued", "device", "back"]


def test_checked_scatter_fails_after_its_check(log):
    src, idx, out = torch.zeros(4, 2), torch.zeros(4, dtype=torch.int64), torch.zeros(1, 2)
    with pytest.raises(_lib.SslaError):
        scatter._run("scatter_max", src, idx, 1, False, out, torch.zeros(1, 2, dtype=torch.int64), True)
    assert log == ["queued", "device", "back"]


def test_kept_where_the_wait_fails(log, monkeypatch):
    def fail(*_):
        raise RuntimeError("device lost")
    monkeypatch.setattr(torch.cuda, "synchronize", fail)
    with pytest.raises(NotImplementedError):
        _recurrent(monkeypatch, NotImplementedError())()
    assert log == ["queued"] and len(_lib.HostWords._lost) == 1


def test_refused_under_capture(log, monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(_lib.SslaError):
        _recurrent(monkeypatch, None)()
    assert log == []


@pytest.mark.gpu
def test_raise_then_call(dev, monkeypatch):
    """A call that raises after its bounds were queued, then others, on two streams."""
    q, k, v, g = (torch.randn(200, 2, 16, device=dev) for _ in range(4))
    cu = torch.tensor([5, 100, 190], device=dev)
    with torch.no_grad():
        want, _ = gla.fused_recurrent_gla(q, k, v, -g.abs(), cu)
        for s in (torch.cuda.current_stream(), torch.cuda.Stream()):
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                with monkeypatch.context() as m:
                    m.setattr(gla, "_recurrent", lambda *_: 1 / 0)
                    with pytest.raises(ZeroDivisionError):
                        gla.fused_recurrent_gla(q, k, v, -g.abs(), cu)
                got, _ = gla.fused_recurrent_gla(q, k, v, -g.abs(), cu)
            torch.cuda.current_stream().wait_stream(s)
            assert got.shape[0] == 185 and torch.equal(got, want)
    assert not _lib.HostWords._lost
