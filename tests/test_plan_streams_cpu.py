"""A plan is on the device when it is handed out: arrays that are copied out of
the build's buffers are waited for, since the plan's next launch may be on
another stream."""

from types import SimpleNamespace

import torch

from flagsparse_amd import _plan


class _Device(torch.Tensor):
    """A host tensor that says it is on a GPU and counts the copies made of it."""

    log = []

    @property
    def is_cuda(self):
        return True

    def clone(self):
        _Device.log.append("copy")
        return super().clone()


def _tensor(n, dtype, held):
    t = torch.zeros(held, dtype=dtype)[:n]
    return t.as_subclass(_Device)


def _finish(monkeypatch, held, n_seg):
    _Device.log = []
    stream = SimpleNamespace(synchronize=lambda: _Device.log.append("wait"))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: stream)
    cfg = _plan.spmm_config(16)
    off = [0, 8, 8, 8, 10 if n_seg else 8]
    rows = _tensor(off[-1], torch.int32, held)
    segments = None
    if n_seg:
        long64 = _tensor(n_seg, torch.int64, held)
        segments = (_tensor(n_seg, torch.int32, held), long64, long64, _tensor(3, torch.int64, held), n_seg)
    indptr = SimpleNamespace(device=torch.device("cpu"))
    plan = _plan._finish_plan(indptr, off[-1], cfg, (rows, off, segments))
    return plan, list(_Device.log)


def test_copied_arrays_are_waited_for(monkeypatch):
    plan, log = _finish(monkeypatch, 1 << 19, 5)
    assert log == ["copy"] * 6 + ["wait"] and plan.seg_begin.untyped_storage().nbytes() == 40
    plan, log = _finish(monkeypatch, 1 << 19, 0)
    assert log == ["copy", "wait"] and plan.rows.untyped_storage().nbytes() == 32


def test_small_buffers_are_kept(monkeypatch):
    assert _finish(monkeypatch, 1000, 5)[1] == [] and _finish(monkeypatch, 1000, 0)[1] == []
